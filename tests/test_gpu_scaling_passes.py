"""The scaling passes at the edges of their tiles (row vectors, column tiles,
row segments of the column maxima) and on views with odd leading dimensions:
the scaled call equals, bit for bit, the same passes done one at a time on the
host (every factor and element update is one correctly rounded operation)
around the unscaled multiply."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _passes(A, B, kind, steps):
    """scaling/scaling.hpp:105-161 in numpy: scaled A and B, r and s."""
    t = A.dtype.type
    r, s = np.ones(A.shape[0], t), np.ones(B.shape[1], t)
    inv = lambda x: np.where(x > 0, 1.0 / np.where(x > 0, x, 1).astype(np.float64), 1.0).astype(t)  # noqa: E731

    def outer():
        nonlocal A, B, r, s
        x, y = np.abs(A).max(axis=1), np.abs(B).max(axis=0)
        A, B = A * inv(x)[:, None], B * inv(y)[None, :]
        r, s = np.where(x > 0, r * x, r), np.where(y > 0, s * y, s)

    def inner():
        nonlocal A, B
        a, b = np.abs(A).max(axis=0).astype(np.float64), np.abs(B).max(axis=1).astype(np.float64)
        ok = (a > 0) & (b > 0)
        z = np.where(ok, np.sqrt(np.where(ok, a, 1) / np.where(ok, b, 1)), 1.0).astype(t)
        A, B = A * (1.0 / z.astype(np.float64)).astype(t)[None, :], B * z[:, None]

    for _ in range(steps):
        for p in {"outside_inside": (outer, inner), "inside_outside": (inner, outer), "inside": (inner,),
                  "outside": (outer,)}[kind]:
            p()
    return A, B, r, s


@pytest.mark.parametrize("kind,steps", [("outside_inside", 1), ("inside_outside", 2), ("inside", 1),
                                        ("outside", 2), ("outside_inside", 0)])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("shape", [(2, 3, 4099), (4099, 3, 2), (17, 16, 1040), (255, 9, 263), (64, 65, 4097),
                                   (3, 8193, 5), (1, 1, 1), (5, 33, 7), (513, 31, 65), (1027, 70, 9), (8195, 3, 33),
                                   (34, 8193, 1030)])
def test_passes_bit_identical(fm, shape, dtype, kind, steps):
    m, k, n = shape
    rng = np.random.default_rng(m + k + n)
    A = (rng.uniform(-1, 1, (m, k)) * 10.0 ** rng.uniform(-3, 3, (m, 1))).astype(dtype)
    B = (rng.uniform(-1, 1, (k, n)) * 10.0 ** rng.uniform(-3, 3, (1, n))).astype(dtype)
    C0 = rng.uniform(-1, 1, (m, n)).astype(dtype)
    A[m // 2] = 0  # a row and a column of zeros keep factor 1
    B[:, n // 2] = 0

    def dev(x, pad):
        p = fm.col_major(torch.zeros((x.shape[0] + pad, x.shape[1]), dtype=torch.from_numpy(x).dtype, device=DEV))
        v = p[pad // 2:pad // 2 + x.shape[0]]
        v.copy_(torch.from_numpy(x))
        return v

    As, Bs, r, s = _passes(A, B, kind, steps)
    for pad, alpha, beta in [(0, 1.0, 0.0), (3, 1.5, -0.5)]:
        P = fm.fastmatmul("strassen", dev(As, 0), dev(Bs, 0), None, 0).cpu().numpy()
        want = (P * r[:, None]) * s[None, :]
        if alpha != 1.0:
            want = dtype(alpha) * want
        if beta != 0.0:
            want = want + dtype(beta) * C0
        C = fm.fastmatmul_scaled("strassen", dev(A, pad), dev(B, pad), dev(C0, pad), 0, alpha=alpha,
                                 beta=beta, scaling=kind, scaling_steps=steps).cpu().numpy()
        assert np.array_equal(C, want), (pad, np.abs(C - want).max())


def test_very_wide_matrices_fit_one_launch(fm):
    """Two rows and 2^27 columns: the lanes of a work group share the columns, so
    a pass takes 2^16 work groups (one per 8 columns would be 2^24, whose 2^32
    threads no launch takes)."""
    n = (1 << 27) + 8
    B = fm.empty(2, n, torch.float32, DEV)
    B.copy_(torch.arange(n, device=DEV, dtype=torch.float32).remainder_(251.0))
    B[1] -= 100.0
    A = fm.col_major(torch.tensor([[2.0, -3.0], [5.0, 7.0]], device=DEV))
    C = fm.fastmatmul_scaled("strassen", A, B, None, 0, scaling_steps=0)
    for i in range(2):  # whole numbers, exact in FP32
        want = A[i, 0] * B[0] + A[i, 1] * B[1]
        assert torch.equal(C[i], want)
