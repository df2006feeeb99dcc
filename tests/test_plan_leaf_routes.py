"""Which leaf kernels a plan gives products that the spread matrix-core loop
cannot take (on the host, through fm_plan_query).

The spread loop needs M of at least one 16-byte vector and K of at least one
16-deep slice; every other product runs on a predicated kernel: 128 x 128
tiles (FmTileCfg 16 in FP64, 5 in FP32) where the launch has enough of them,
64 x 64 (FmTileCfg 1) where a larger tile would be mostly empty.
"""
import pytest
import torch

import fastmm

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
