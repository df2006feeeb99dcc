"""Dynamic-peeling products at the edges of their kernels' tiles: every
remainder of every block split the algorithms have, in each dimension.

A's (then B's) rows and columns inside the block split are zero, so the
recursion contributes exact zeros and, on integer data, every element of C is
an exact integer: the comparison is bit for bit, whatever the order of the
sums.  With A's zeros the bottom strip runs over all of K, with B's the right
strip does; the K update has all its data in both."""
import os
import subprocess

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

SPLITS = {"strassen": (2, 2, 2), "classical333_27_81": (3, 3, 3), "grey424_26_206": (4, 2, 4),
          "grey522_18_99": (5, 2, 2), "smirnov633_40_960": (6, 3, 3), "smirnov363_40_960": (3, 6, 3),
          "smirnov336_40_960": (3, 3, 6)}


def _check(fm, alg, m, k, n, dtype, alpha, beta, seed):
    sm, sk, sn = SPLITS[alg]
    rng = np.random.default_rng(seed)
    dev = lambda x: fm.col_major(torch.from_numpy(np.asfortranarray(x)).to(DEV))  # noqa: E731
    for zeros_in_a in (True, False):
        A = rng.integers(-8, 9, (m, k)).astype(dtype)
        B = rng.integers(-8, 9, (k, n)).astype(dtype)
        C0 = rng.integers(-8, 9, (m, n)).astype(dtype)
        if zeros_in_a:  # the core's products vanish
            A[:m - m % sm, :k - k % sk] = 0
        else:
            B[:k - k % sk, :n - n % sn] = 0
        want = alpha * (A.astype(np.float64) @ B.astype(np.float64)) + beta * C0.astype(np.float64)
        C = fm.fastmatmul(alg, dev(A), dev(B), dev(C0), 1, alpha=alpha, beta=beta).double().cpu().numpy()
        assert np.array_equal(C, want), (alg, m, k, n, zeros_in_a, np.argwhere(C != want)[:4])


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("alg", sorted(SPLITS))
def test_every_remainder(fm, alg, dtype):
    sm, sk, sn = SPLITS[alg]
    for r in range(1, max(SPLITS[alg])):
        m, k, n = 48 * sm + r % sm, 40 * sk + r % sk, 24 * sn + r % sn
        _check(fm, alg, m, k, n, dtype, 2.0, -3.0, r)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("shape", [
    (3, 3, 3),            # single rows, columns and K
    (17, 255, 31),        # one past a strip's row tile, one short of a segment round
    (257, 1027, 65),      # one past the update's rows, a wave's K round and columns
    (33, 129, 1031),      # many bottom-strip tiles
    (1031, 65, 19),
])
def test_tile_edges(fm, shape, dtype):
    for alpha, beta in [(1.0, 0.0), (-1.0, 2.0)]:
        _check(fm, "strassen", *shape, dtype, alpha, beta, sum(shape))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("k", [2, 5, 8, 9, 16, 17, 33, 64, 65, 127, 128, 129, 257])
def test_strips_of_a_short_k(fm, k, dtype):
    """K segments and lanes of the strips: one, as many as K fills, and all of
    them (the limits are 8 and 4 values of K per segment and lane), with rows
    and columns one past, and one short of, every tile that goes with them."""
    for m, n in [(257, 1031), (1025, 513), (33, 63), (255, 129)]:
        _check(fm, "strassen", m, k, n, dtype, -1.0, 2.0, k)
    _check(fm, "smirnov336_40_960", 3 * 90 + 2, k + 1, 6 * 60 + 5, dtype, 1.0, 0.0, k)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("alg,shape", [
    ("strassen", (2056, 1027, 2052)),             # K remainder alone, 16-byte rows in the W stage
    ("grey522_18_99", (2063, 1027, 2051)),        # every remainder, odd rows
    ("smirnov363_40_960", (1230, 1025, 1231)),    # K remainder of 5
])
def test_k_remainder_in_the_w_stage_of_larger_products(fm, alg, shape, dtype):
    """Above the size where W shares its launch with the strips."""
    for alpha, beta in [(1.0, 0.0), (2.0, -3.0)]:
        _check(fm, alg, *shape, dtype, alpha, beta, 5)


def test_stages_apart_and_together_give_the_same_bits(fm):
    """One problem's S and T, and W, K remainder and strips, share launches
    where small; a batch of two problems runs each stage and the peeling
    apart."""
    rng = np.random.default_rng(11)
    dev = lambda x: fm.col_major(torch.from_numpy(np.asfortranarray(x)).to(DEV))  # noqa: E731
    for alg, steps, (m, k, n) in [("strassen", 2, (259, 262, 133)), ("grey424_26_206", 1, (403, 205, 303)),
                                  ("grey333_23_152", 2, (190, 187, 185)), ("smirnov633_40_960", 1, (131, 65, 98)),
                                  ("strassen", 1, (4099, 515, 1030))]:
        for dt in (np.float64, np.float32):
            A, B, C0 = (dev((rng.random(s) * 2 - 1).astype(dt)) for s in ((m, k), (k, n), (m, n)))
            one = fm.fastmatmul(alg, A, B, C0.clone(), steps, alpha=1.5, beta=0.5)
            probs = [{"A": A, "B": B, "C": C0.clone(), "alg": alg, "num_steps": steps, "alpha": 1.5, "beta": 0.5}
                     for _ in range(2)]
            fm.Batch(probs, graph=False).run()
            torch.cuda.synchronize()
            assert torch.equal(one, probs[0]["C"]) and torch.equal(one, probs[1]["C"]), (alg, dt)


def test_peeling_in_a_batch_of_unequal_problems(fm):
    """Products of several shapes in one launch (found by the search, not by
    division), each equal to its own call bit for bit."""
    rng = np.random.default_rng(9)
    dev = lambda x: fm.col_major(torch.from_numpy(np.asfortranarray(x)).to(DEV))  # noqa: E731
    probs, single = [], []
    for alg, (m, k, n) in [("strassen", (131, 77, 95)), ("grey522_18_99", (204, 301, 65)),
                           ("strassen", (64, 65, 64)), ("strassen", (66, 64, 131))]:
        A, B, C0 = (dev(rng.random(s) * 2 - 1) for s in ((m, k), (k, n), (m, n)))
        probs.append({"A": A, "B": B, "C": C0.clone(), "alg": alg, "num_steps": 1, "alpha": 1.5, "beta": 0.5})
        single.append(fm.fastmatmul(alg, A, B, C0.clone(), 1, alpha=1.5, beta=0.5))
    fm.Batch(probs, graph=False).run()
    torch.cuda.synchronize()
    for p, s in zip(probs, single):
        assert torch.equal(p["C"], s)


@pytest.fixture(scope="module")
def thin_k_probe(tmp_path_factory):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    exe = str(tmp_path_factory.mktemp("thin") / "thin_k_probe")
    lib = os.path.join(root, "fast-matmul_amd", "fastmm")
    subprocess.check_call(
        ["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(root, "include"),
         "-I", os.path.join(root, "fast-matmul_amd", "csrc"), "-I", "/opt/rocm/include",
         os.path.join(root, "tests", "cpp", "thin_k_probe.cpp"), "-o", exe, "-L", lib, "-lfastmm",
         "-L", "/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath," + lib + ":/opt/rocm/lib"])
    return exe


@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_k_update_of_a_split_finer_than_the_tables(fm, thin_k_probe, dtype):
    """A K remainder of 5 (the last with a kernel of its own), and beyond it,
    where the update loops over K: no shipped table splits K so finely, so
    the kernel is called by itself."""
    for M, N, K, beta in [(300, 37, 5, 1), (300, 37, 6, 1), (257, 16, 9, 0), (1, 1, 20, 1), (255, 33, 31, -2)]:
        subprocess.check_call([thin_k_probe, dtype, str(M), str(N), str(K), str(beta)], timeout=60)
