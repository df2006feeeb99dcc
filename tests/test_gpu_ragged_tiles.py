"""The spread leaf kernels on products of any size and alignment: views into
NaN-filled parents at odd offsets with odd leading dimensions, at every
remainder of the K slice and of the row vector.

Integer data: every partial sum is an exact integer, so the result does not
depend on the order of k and the comparison is bit for bit; a NaN that
reaches an accumulator, or an element outside the view of C that changes,
shows as a difference."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
CFGS = [-1, 1, 2, 3, 32, 33, 34]  # -1: the plan's own choice (32 x 32 tiles for these sizes)


@pytest.fixture(autouse=True)
def _reset(fm):
    yield
    fm.set_gemm_tile(-1)


def _view(fm, x, off, pad):
    """x as a view at row and column `off` of a NaN-filled column-major parent."""
    p = np.full((x.shape[0] + off + pad, x.shape[1] + 2 * off), np.nan, dtype=x.dtype)
    p[off:off + x.shape[0], off:off + x.shape[1]] = x
    t = fm.col_major(torch.from_numpy(np.asfortranarray(p)).to(DEV))
    return t, t[off:off + x.shape[0], off:off + x.shape[1]]


def _check(fm, m, k, n, dtype, off, pad, alpha=1.0, beta=0.0):
    rng = np.random.default_rng(m * 7919 + k * 31 + n)
    A = rng.integers(-8, 9, (m, k)).astype(dtype)
    B = rng.integers(-8, 9, (k, n)).astype(dtype)
    C = rng.integers(-8, 9, (m, n)).astype(dtype)
    (_, a), (_, b), (pc, c) = _view(fm, A, off, pad), _view(fm, B, off, pad), _view(fm, C, off, pad)
    fm.gemm(a, b, c, alpha, beta)
    want = alpha * (A.astype(np.float64) @ B.astype(np.float64)) + beta * C.astype(np.float64)
    parent = pc.double().cpu().numpy()
    assert np.array_equal(parent[off:off + m, off:off + n], want), (m, k, n)
    parent[off:off + m, off:off + n] = np.nan
    assert np.isnan(parent).all()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("cfg", CFGS)
def test_every_k_remainder(fm, cfg, dtype):
    fm.set_gemm_tile(cfg)
    # (slices of 16: whole, partial and both parities of the loop's trips)
    for k in list(range(16, 34)) + [47, 63, 65, 97]:
        _check(fm, 37, k, 29, dtype, 1, k % 3)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_every_k_remainder_of_the_32_deep_tile(fm, dtype):
    """The 32 x 32 tile has slices of 32 and is the plan's choice only: every
    remainder of its slice behind five and six of them, so that the loop's
    body, both of its halves and the iterations before a partial slice all run."""
    td = torch.float64 if dtype is np.float64 else torch.float32
    for k in range(160, 224):
        assert fm.plan_info("strassen", 37, k, 29, 0, dtype=td)["leaf"][0]["cfg"] == 35
        _check(fm, 37, k, 29, dtype, 1, k % 3)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("cfg", CFGS)
def test_row_and_column_edges(fm, cfg, dtype):
    fm.set_gemm_tile(cfg)
    for m in (1, 2, 3, 4, 5, 31, 33, 63, 65, 127, 128, 129, 130, 131):
        _check(fm, m, 50, 2 * m + 1, dtype, 1, 0)
    for n in (1, 31, 33, 95, 97, 127, 129, 255, 257):
        _check(fm, 66, 35, n, dtype, 0, 1, 2.0, -3.0)
    # aligned views with partial tiles, and whole tiles at an odd offset
    _check(fm, 260, 64, 200, dtype, 4, 4)
    _check(fm, 256, 64, 256, dtype, 1, 1)
