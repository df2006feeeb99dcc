"""Which leaf kernels a plan gives products that the spread matrix-core loop
cannot take (on the host, through fm_plan_query).

The spread loop needs M of at least one 16-byte vector and K of at least one
16-deep slice; every other product runs on a predicated kernel: 128 x 128
tiles (FmTileCfg 16 in FP64, 5 in FP32) where the launch has enough of them,
64 x 64 (FmTileCfg 1) where a larger tile would be mostly empty.
"""
import os
import subprocess

import pytest
import torch

import fastmm

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EDGE = {torch.float64: 16, torch.float32: 5}


def _leaf(m, k, n, dtype, steps=0):
    return fastmm.plan_info("strassen", m, k, n, steps, dtype=dtype)["leaf"][0]["cfg"]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("k", [1, 4, 14, 15])
def test_shallow_products_take_the_large_predicated_tile(k, dtype):
    assert _leaf(4096, k, 4096, dtype) == EDGE[dtype]
    assert _leaf(16384, k, 16384, dtype) == EDGE[dtype]
    assert _leaf(8192, 2 * k, 8192, dtype, 1) == EDGE[dtype]  # seven leaves of 4096 x k x 4096


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_single_rows_keep_the_small_predicated_tile(dtype):
    # one row: half of a 64-row tile's work is spared against a 128-row one
    for n in (4096, 1000000):
        assert _leaf(1, 4096, n, dtype) == 1
    # and the spread loop takes everything else
    assert _leaf(4096, 16, 4096, dtype) not in (1, EDGE[dtype])
    assert _leaf(4, 4096, 4096, dtype) not in (EDGE[dtype],)


# ---- several problems in one launch sequence ------------------------------------
@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    """run(dtype, problems): the launches of a batch's plan, as tests/cpp/plan_probe.cpp prints them."""
    exe = str(tmp_path_factory.mktemp("plan") / "plan_probe")
    lib = os.path.join(ROOT, "fast-matmul_amd", "fastmm")
    subprocess.check_call(
        ["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROOT, "include"),
         "-I", os.path.join(ROOT, "fast-matmul_amd", "csrc"), "-I", "/opt/rocm/include",
         os.path.join(ROOT, "tests", "cpp", "plan_probe.cpp"), "-o", exe, "-L", lib, "-lfastmm",
         "-L", "/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath," + lib + ":/opt/rocm/lib"])

    def run(dtype, problems):
        args = [",".join(str(v) for v in p) for p in problems]
        out = subprocess.check_output([exe, dtype] + args, text=True)
        return [l.split()[:1] + [int(v) for v in l.split()[1:]] for l in out.splitlines()]

    return run


def _gemms(launches):
    """{"cfg", "any", "full", "products", "tiles", "k"} of each leaf launch."""
    return [dict(zip(("cfg", "any", "full", "products", "tiles", "k"), l[1:])) for l in launches if l[0] == "gemm"]


def _spread(launches):
    return [g for g in launches if g["any"] or g["full"]]


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("odd", [(4096, 8, 4096), (1, 2048, 2048)])
def test_one_odd_problem_leaves_the_others_their_kernels(probe, dtype, odd):
    # 63 large problems of ragged sizes and one that the spread loop cannot take
    # (in FP32 one of the 63 has a bottom strip of 3 rows, less than a vector)
    big = [(1000 + 37 * i, 1500 + 11 * (i % 7), 900 + 53 * i) for i in range(63)]
    alone = _gemms(probe(dtype, big))
    mixed = _gemms(probe(dtype, big[:20] + [odd] + big[20:]))
    assert len(_spread(alone)) == 2 and _spread(mixed) == _spread(alone)
    rest = [g for g in mixed if g not in _spread(mixed)]
    assert len(rest) == 1 and rest[0]["products"] == (1 if dtype == "f64" else 2)


@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_one_row_strip_leaves_the_other_strips_their_kernels(probe, dtype):
    # cores of whole tiles with right strips 40 columns wide, and one problem
    # whose bottom strip is one row
    big = [(2048, 2048, 2048 + 40)] * 200
    alone = _gemms(probe(dtype, big + [(2048, 2048, 2048)]))
    mixed = _gemms(probe(dtype, big + [(2049, 2048, 2048)]))
    assert [g["products"] for g in _spread(alone)] == [201, 200]
    for g, h in zip(_spread(mixed), _spread(alone)):
        assert (g["cfg"], g["products"], g["tiles"]) == (h["cfg"], h["products"], h["tiles"])
    assert len(_spread(mixed)) == 2
    rest = [g for g in mixed if g not in _spread(mixed)]
    assert [g["products"] for g in rest] == [1]


def test_an_odd_problem_that_would_only_wait_stays(probe):
    # 12 such problems: alone, the one row's chain over K would take longer than
    # all strips do beside it, so they share its launch
    g = _gemms(probe("f64", [(2048, 2048, 2048 + 40)] * 12 + [(2049, 2048, 2048)]))
    assert [x["products"] for x in g] == [13, 13]


@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_only_odd_problems_share_one_launch(probe, dtype):
    g = _gemms(probe(dtype, [(500, 3, 500), (1, 300, 700), (900, 15, 100)]))
    assert len(g) == 1 and not g[0]["any"] and g[0]["products"] == 3


# ---- peeled strips ----------------------------------------------------------------
def _strip_tiles(launches):
    """Work groups of the launches of peeled strips on their own."""
    return [l[2] for l in launches if l[0] == "thin"]


@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_strips_of_a_short_k_take_few_work_groups(probe, dtype):
    # two problems, so that the strips run in a launch of their own; K = 8 is one
    # segment of 256 rows (two lanes of 512 columns)
    for m, k, n, groups in [(1000001, 8, 4, 0), (1000000, 8, 5, 3907), (5, 8, 1000000, 1954)]:
        t = _strip_tiles(probe(dtype, [(m, k, n, "strassen", 1), (m, k, n, "strassen", 1)]))
        one_row = 1 if m == 1000001 else 0  # its bottom row: one work group
        assert t == [2 * (groups or one_row)]


def test_strips_of_long_matrices_fit_one_launch(probe):
    # a launch holds fewer than 2^32 threads, 2^24 of these work groups
    for p in [(1 << 28, 2, 3), ((1 << 29) + 4, 6, 3), (3, 2, 1 << 30)]:
        t = _strip_tiles(probe("f64", [p + ("strassen", 1), (64, 64, 65, "strassen", 1)]))
        assert t and max(t) < 1 << 24


# ---- large launches of shallow products --------------------------------------------
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_large_shallow_launches_leave_the_smallest_tile(dtype):
    # seven leaves of 150000 x 32 x 32: 128 x 64 tiles (FmTileCfg 2), not 32 x 32 (35)
    assert _leaf(300000, 64, 64, dtype, 1) == 2
    assert _leaf(300000, 64, 16, dtype, 1) == 2
    assert _leaf(64, 64, 300000, dtype, 1) in (1, 3)
    # deeper, or few tiles: the smallest tile still
    assert _leaf(300000, 512, 16, dtype, 1) == 35
    assert _leaf(64, 64, 64, dtype) == 35
    if dtype == torch.float64:  # 64 x 64 tiles up to K = 64, 64 x 128 (3) beyond
        assert [_leaf(128, 2 * k, 300000, dtype, 1) for k in (16, 64, 256)] == [1, 1, 3]


# ---- depth-first problems of a batch -------------------------------------------------
def _peeling_products(launches):
    """Peeling products in launches of their own and in W stages (the K updates among them)."""
    return sum(l[1] for l in launches if l[0] == "thin") + sum(l[4] for l in launches if l[0] == "stage")


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("dfs", [0, 1, 2])
def test_grouped_problems_keep_every_peeling_product(probe, dtype, dfs):
    # remainders of every dimension at both levels; a depth-first child's W
    # stage adds its K remainder itself, also where the same stage of another
    # problem stands beside it
    ps = [(2 * (2 * 130 + 1) + 1, 2 * (2 * 90 + 1) + 1, 2 * (2 * 70 + 1) + 1, "strassen", 2, dfs),
          (2 * (2 * 60 + 1) + 1, 2 * (2 * 80 + 1) + 1, 2 * (2 * 50 + 1) + 1, "strassen", 2, dfs)]
    alone = [_peeling_products(probe(dtype, [p])) for p in ps]
    assert alone == [3 + 7 * 3, 3 + 7 * 3]
    assert _peeling_products(probe(dtype, ps)) == sum(alone)
    # K remainders alone: the W stages that add them have no strips beside them
    ps = [(4 * m, 2 * (2 * k + 1), 4 * n, "strassen", 2, dfs) for m, k, n in [(130, 90, 70), (60, 80, 50)]]
    alone = [_peeling_products(probe(dtype, [p])) for p in ps]
    assert alone == [7, 7]
    assert _peeling_products(probe(dtype, ps)) == sum(alone)


# ---- stage-written slice planes ------------------------------------------------------
def _split(alg, m, k, n, fusion):
    fastmm.set_stage_fusion(fusion)
    try:
        return fastmm.plan_info(alg, m, k, n, 2, dtype=torch.float32, mode="split_bf16")
    finally:
        fastmm.set_stage_fusion(True)


@pytest.mark.parametrize("alg,m,k,n", [("strassen", 1 << 18, 4, 4), ("strassen", 1 << 20, 8, 4),
                                       ("grey223_11_50", 254665, 17, 387), ("grey234_20_144", 35873, 9, 49),
                                       ("grey232_11_50", 244620, 74, 496), ("grey332_15_103", 604153, 9, 348),
                                       ("strassen", 1 << 16, 128, 4), ("strassen", 3448, 3448, 3448)])
def test_padded_planes_take_no_more_workspace(alg, m, k, n):
    """Planes written by the S/T stage, padded to whole tiles and slices,
    against planes cut from FP32 operands by the separate pass."""
    assert _split(alg, m, k, n, 1)["workspace_bytes"] <= _split(alg, m, k, n, 2)["workspace_bytes"]


def test_padded_planes_stay_within_32_bit_counts():
    # leaves of 2^27 x 1: 2^32 elements with K padded to a slice; the separate pass prepares them
    assert _split("strassen", 1 << 29, 4, 4, 1)["prep_bytes"] == _split("strassen", 1 << 29, 4, 4, 2)["prep_bytes"]
    # leaves of 2^25 + 256 rows and 33 columns: past 2^31 with K padded to two slices
    m = 4 * ((1 << 25) + 256)
    assert _split("strassen", m, 4 * 33, 4, 1)["prep_bytes"] == _split("strassen", m, 4 * 33, 4, 2)["prep_bytes"]
    # and the path itself is still taken
    assert _split("strassen", 3448, 3448, 3448, 1)["prep_bytes"] < _split("strassen", 3448, 3448, 3448, 2)["prep_bytes"]


# ---- splits finer than any shipped table's -------------------------------------------
@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("split", [(9, 2, 2), (2, 9, 2), (2, 2, 9), (10, 11, 17), (2, 8, 2), (6, 6, 6), (7, 7, 7)])
@pytest.mark.parametrize("scale", [5, 400])
def test_remainders_of_fine_splits_are_all_peeled(probe, dtype, split, scale):
    """The peeling products of one level cover C's strips once each, in pieces
    the kernels take, and its core by one update of the whole K remainder."""
    m, k, n = (s * scale + s - 1 for s in split)
    if scale == 400 and split == (10, 11, 17):
        m, k, n = (s * 40 + s - 1 for s in split)
    launches = probe(dtype, [(m, k, n, "blocks:%dx%dx%d" % split, 1)])
    cm, ck, cn = (v // s * s for v, s in zip((m, k, n), split))
    seen = [[0] * n for _ in range(m)] if m * n < 200000 else None
    area = updates = 0
    at, fused = None, 0
    for l in launches:
        if l[0] == "stage":
            fused = l[3]
        if l[0] != "peel":
            at = l
            continue
        kind, M, N, K, off, ld = l[1:]
        assert ld == m
        if kind == 0:
            updates += 1
            assert (M, N, K, off) == (cm, cn, k - ck, 0)
            # added by the W stage up to a split its kernel is built for, else in a launch after it
            assert (at[0] == "stage") == (split[1] <= 6)
            continue
        assert K == k and (M if kind == 2 else N) <= 5
        i0, j0 = off % ld, off // ld
        area += M * N
        if seen is not None:
            for i in range(i0, i0 + M):
                for j in range(j0, j0 + N):
                    seen[i][j] += 1
    assert updates == (1 if k > ck else 0) and fused == (updates if split[1] <= 6 else 0)
    assert area == m * n - cm * cn
    if seen is not None:
        assert all(seen[i][j] == (0 if i < cm and j < cn else 1) for i in range(m) for j in range(n))
