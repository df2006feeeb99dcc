"""Performance cases of the fast multiply.

Each case is one call that a program makes again and again: inputs resident
in HBM, column-major, a preallocated C (and, where such a program keeps one,
a plan or a batch), and one pass through the public entry points of
``fastmm``.  Sizes are those of the reference's test and benchmark shapes
(tests/matmul_tests.cpp:140-145, data/README.md) and of this repository's
own benchmark workloads; ``draw`` spreads further cases over the same ranges.
"""
from __future__ import annotations

import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "fast-matmul_amd"))

import fastmm  # noqa: E402

DEV = "cuda:0"
_DT = {"f64": torch.float64, "f32": torch.float32}


def _case(entry, alg, steps, m, k, n, dtype="f64", mode="plain", alpha=1.0, beta=0.0, dist="u11", **kw):
    c = {"entry": entry, "alg": alg, "steps": steps, "m": m, "k": k, "n": n, "dtype": dtype,
         "mode": mode, "alpha": alpha, "beta": beta, "dist": dist}
    c.update(kw)
    return c


def listed():
    return [
        # the smallest call: the README's known-answer product, where launches
        # and host work count (dimensions divide by neither the block split
        # nor the vector width)
        dict(_case("call", "strassen", 1, 257, 500, 55, dist="u01"), name="small_257x500x55"),
        # C := alpha A B + beta C at a test shape that peels in every dimension
        dict(_case("call", "grey522_18_99", 1, 1007, 400, 679, alpha=1.5, beta=-0.5, dist="u01"),
             name="alpha_beta_1007x400x679"),
        # an ordinary square multiply through a kept plan and workspace, as a
        # serving loop runs it
        dict(_case("plan", "strassen", 1, 2048, 2048, 2048), name="plan_strassen_2048"),
        # the 4000-scale test shapes: two levels, peeling at both
        dict(_case("call", "grey333_23_152", 2, 4009, 2800, 2489), name="ragged_4009x2800x2489"),
        # the headline benchmark
        dict(_case("call", "grey424_26_206", 2, 8192, 8192, 8192), name="square_8192"),
        # tall times square (the reference's tssquare workload)
        dict(_case("call", "grey424_26_206", 1, 131072, 2400, 2400), name="tall_131072x2400x2400"),
        # outer-product shape (the reference's matrix-addition study)
        dict(_case("call", "grey424_26_206", 1, 9000, 1600, 9000), name="outer_9000x1600x9000"),
        # single precision at a round decimal size
        dict(_case("call", "strassen", 2, 5000, 5000, 5000, dtype="f32"), name="f32_5000"),
        # single precision on split-bf16 leaves, the largest square workload
        dict(_case("call", "strassen", 2, 16384, 16384, 16384, dtype="f32", mode="split_bf16"),
             name="split_16384"),
        # diagonal scaling around a single-precision multiply of badly scaled data
        dict(_case("scaled", "strassen", 1, 4096, 4096, 4096, dtype="f32", dist="skew"), name="scaled_f32_4096"),
        # double precision on int8-digit leaves
        dict(_case("call", "smirnov333_23_139", 2, 13824, 13824, 13824, mode="ozaki_int8"), name="digits_13824"),
        # many uneven single-precision products in one replayed launch sequence
        dict(_case("batch", "auto", 0, 4096, 4096, 4096, dtype="f32", count=64, low=512, step=64), name="batch_64_uneven"),
    ]


# ---- further cases of the same ranges -----------------------------------------
_ALGS = ["strassen", "grey424_26_206", "grey423_20_144", "grey333_23_152", "smirnov333_23_139",
         "grey522_18_99", "hk332_15_94"]


def _size(rng, lo, hi):
    """Log-uniform on [lo, hi]: any integer, a multiple of 8 or (from 512) of 64."""
    v = int(round(lo * (hi / lo) ** rng.random()))
    q = rng.choice([1, 8, 64]) if v >= 512 else rng.choice([1, 8])
    return max(lo, v // q * q)


def draw(rng):
    family = rng.choice(["small", "alpha_beta", "plan", "ragged", "square", "tall", "outer", "f32",
                         "split", "scaled", "digits", "batch"])
    if family == "small":
        alg = rng.choice(_ALGS)
        return _case("call", alg, 1, _size(rng, 100, 700), _size(rng, 100, 600), _size(rng, 50, 700),
                     dtype=rng.choice(["f64", "f64", "f32"]), dist="u01")
    if family == "alpha_beta":
        return _case("call", rng.choice(_ALGS), rng.choice([1, 2]), _size(rng, 600, 3000), _size(rng, 200, 2000),
                     _size(rng, 300, 3000), alpha=rng.choice([1.0, 1.5, -1.25]), beta=rng.choice([0.5, -0.5]),
                     dist="u01")
    if family == "plan":
        s = _size(rng, 1000, 4096)
        return _case("plan", rng.choice(["strassen", "grey423_20_144", "smirnov333_23_139"]), 1, s, s, s,
                     dtype=rng.choice(["f64", "f32"]))
    if family == "ragged":
        return _case("call", rng.choice(_ALGS), rng.choice([1, 2]), rng.randint(2000, 4500), rng.randint(2000, 4500),
                     rng.randint(2000, 4500), dtype=rng.choice(["f64", "f32"]))
    if family == "square":
        s = _size(rng, 4096, 10000)
        return _case("call", rng.choice(["strassen", "grey424_26_206", "smirnov333_23_139"]), rng.choice([1, 2]),
                     s, s, s)
    if family == "tall":
        w = _size(rng, 800, 2400)
        return _case("call", rng.choice(["grey424_26_206", "grey423_20_144"]), rng.choice([1, 2]),
                     _size(rng, 10000, 131072), w, w)
    if family == "outer":
        s = _size(rng, 3000, 9000)
        return _case("call", rng.choice(["grey424_26_206", "hk332_15_94"]), 1, s, _size(rng, 800, 1600), s)
    if family == "f32":
        s = _size(rng, 2000, 8192)
        return _case("call", rng.choice(["strassen", "grey423_20_144"]), rng.choice([1, 2]), s, s, s, dtype="f32")
    if family == "split":
        s = _size(rng, 2048, 16384)
        return _case("call", rng.choice(["strassen", "grey424_26_206"]), rng.choice([1, 2]), s, s, s, dtype="f32",
                     mode="split_bf16")
    if family == "scaled":
        s = _size(rng, 1000, 4096)
        return _case("scaled", "strassen", rng.choice([1, 2]), s, s, s, dtype=rng.choice(["f32", "f64"]), dist="skew")
    if family == "digits":
        s = _size(rng, 3000, 13824)
        return _case("call", rng.choice(["strassen", "smirnov333_23_139"]), rng.choice([1, 2]), s, s, s,
                     mode="ozaki_int8")
    hi = rng.choice([1024, 2048, 4096])
    return _case("batch", "auto", 0, hi, hi, hi, dtype="f32", count=rng.randint(12, 64), low=rng.choice([256, 512]),
                 step=rng.choice([64, 8, 1]), mode=rng.choice(["plain", "split_bf16"]))


# ---- inputs ---------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _matrix(g, rows, cols, dtype, dist):
    """A column-major rows x cols matrix."""
    x = torch.rand((cols, rows), generator=g, device=DEV, dtype=dtype)
    if dist != "u01":
        x = x * 2 - 1
    return x.t()


def _inputs(case, seed):
    g, dt = _gen(seed), _DT[case["dtype"]]
    m, k, n, dist = case["m"], case["k"], case["n"], case["dist"]
    A, B = _matrix(g, m, k, dt, dist), _matrix(g, k, n, dt, dist)
    if dist == "skew":  # rows of A and columns of B over six orders of magnitude
        A = A * 10.0 ** (torch.rand((m, 1), generator=g, device=DEV, dtype=dt) * 6 - 3)
        B = B * 10.0 ** (torch.rand((1, n), generator=g, device=DEV, dtype=dt) * 6 - 3)
    C = _matrix(g, m, n, dt, dist) if case["beta"] != 0.0 else fastmm.empty(m, n, dt, DEV)
    return fastmm.col_major(A), fastmm.col_major(B), C


def _batch_shapes(case):
    """The shapes of a batch: fixed by the case, from [low, m] in steps of ``step``."""
    vals = list(range(case["low"], case["m"] + 1, case["step"]))
    state, out = 0xC3 + case["count"] * 7919 + case["m"], []
    for _ in range(case["count"]):
        s = []
        for _ in range(3):
            state = (state * 6364136223846793005 + 1442695040888963407) % (1 << 64)
            s.append(vals[(state >> 33) % len(vals)])
        out.append(tuple(s))
    return out


def _batch_inputs(case, seed):
    g, dt = _gen(seed), _DT[case["dtype"]]
    return [{"A": _matrix(g, m, k, dt, case["dist"]), "B": _matrix(g, k, n, dt, case["dist"]),
             "C": fastmm.empty(m, n, dt, DEV)} for m, k, n in _batch_shapes(case)]


def prepare(case, seed):
    if case["entry"] == "batch":
        probs = _batch_inputs(case, seed)
        return {"case": case, "batch": fastmm.Batch(probs, mode=case["mode"], graph=True),
                "C": [p["C"] for p in probs]}
    A, B, C = _inputs(case, seed)
    st = {"case": case, "A": A, "B": B, "C": C}
    if case["entry"] == "plan":
        st["plan"] = fastmm.Plan(case["alg"], case["m"], case["k"], case["n"], case["steps"],
                                 dtype=_DT[case["dtype"]], mode=case["mode"])
        st["ws"] = torch.empty(st["plan"].workspace_bytes(), dtype=torch.uint8, device=DEV)
    return st


def run(state):
    c = state["case"]
    if c["entry"] == "batch":
        state["batch"].run()
        return state["C"]
    if c["entry"] == "plan":
        return state["plan"].run(state["A"], state["B"], state["C"], workspace=state["ws"])
    if c["entry"] == "scaled":
        return fastmm.fastmatmul_scaled(c["alg"], state["A"], state["B"], state["C"], c["steps"], mode=c["mode"])
    return fastmm.fastmatmul(c["alg"], state["A"], state["B"], state["C"], c["steps"], alpha=c["alpha"],
                             beta=c["beta"], mode=c["mode"])


# ---- what a pass cannot do without ------------------------------------------------
def _work(alg, steps, m, k, n, es, beta):
    """The multiplications of the named algorithm at this depth (leaf products
    and, per level, the peeled rows and columns); A and B read, C written."""
    flops, nodes, mm, kk, nn = 0.0, 1.0, m, k, n
    if alg != "auto":
        a = fastmm.alg(alg)
        for _ in range(steps):
            bm, bk, bn = mm // a.dims[0], kk // a.dims[1], nn // a.dims[2]
            core = float(bm * a.dims[0]) * (bk * a.dims[1]) * (bn * a.dims[2])
            flops += nodes * 2.0 * (float(mm) * kk * nn - core)
            nodes *= a.rank
            mm, kk, nn = bm, bk, bn
    flops += nodes * 2.0 * mm * kk * nn
    return flops, float(es) * (m * k + k * n + m * n * (2 if beta else 1))


def work(case):
    es = 8 if case["dtype"] == "f64" else 4
    if case["entry"] == "batch":
        parts = [_work("auto", 0, m, k, n, es, 0) for m, k, n in _batch_shapes(case)]
        return {"flops": sum(p[0] for p in parts), "bytes": sum(p[1] for p in parts)}
    f, b = _work(case["alg"], case["steps"], case["m"], case["k"], case["n"], es, case["beta"] != 0.0)
    return {"flops": f, "bytes": b}


# Relative 2-norm error against the 64-bit product, four times the largest seen
# over the listed cases and 240 drawn ones, by data type and depth; the second
# figure is for <4,2,4;26>, whose coefficient sums amplify rounding more.
# Split-bf16 leaves (FP32) and int8-digit leaves (FP64) stay within the plain
# figures.
_REL = {
    ("f32", 0): (4.6e-6, 4.6e-6),
    ("f32", 1): (1.4e-5, 1.8e-5),
    ("f32", 2): (2.7e-5, 5.0e-5),
    ("f64", 1): (2.0e-14, 3.3e-14),
    ("f64", 2): (3.2e-14, 8.0e-14),
}
# Badly scaled data: entries far below the result's root mean square carry the
# error of the large rows and columns they are combined with.
_MAX_SKEW = {"f32": 1.0e-3, "f64": 2.0e-12}


def tolerance(case):
    t = {"rel": _REL[(case["dtype"], case["steps"])][1 if "424" in case["alg"] else 0]}
    if case["dist"] == "skew":
        t["max"] = _MAX_SKEW[case["dtype"]]
    return t


def _product(A, B):
    """A B in 64 bits, by torch."""
    return torch.matmul(B.double().t(), A.double().t()).t()


def exact(case, seed):
    if case["entry"] == "batch":
        return [_product(p["A"], p["B"]) for p in _batch_inputs(case, seed)]
    A, B, C = _inputs(case, seed)
    P = _product(A, B)
    if case["beta"] != 0.0:
        return case["alpha"] * P + case["beta"] * C.double()
    return case["alpha"] * P
