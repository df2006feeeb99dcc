"""Stage-written slice planes of leaves that are not whole tiles: the last
two-level S/T stage pads the planes with zeros (rows to 256, K to 32), and the
result equals the separate preparation's bit for bit, at every lane width of
the stage kernels (4, 2 and 1; staged through LDS or not) and one to many
rows and k short of or past the padding."""
import numpy as np
import pytest
import torch

from cases import make_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("alg,steps,unit,leaf,fused", [
    ("strassen", 2, (4, 4, 4), (521, 353, 515), True),
    ("strassen", 2, (4, 4, 4), (255, 1024, 256), True),     # rows short, K whole
    ("strassen", 2, (4, 4, 4), (256, 1057, 255), True),     # K past, columns short
    ("strassen", 2, (4, 4, 4), (1025, 193, 129), True),     # S planes only
    ("strassen", 2, (4, 4, 4), (128, 250, 1100), True),     # T planes only
    ("strassen", 2, (4, 4, 4), (130, 33, 130), False),      # too few lanes
    ("strassen", 3, (8, 8, 8), (261, 513, 257), True),
    ("grey424_26_206", 2, (16, 4, 16), (137, 1030, 131), True),
    ("grey223_11_50", 2, (4, 4, 9), (130, 1055, 140), True),
    ("smirnov333_23_139", 2, (9, 9, 9), (150, 1025, 170), True),
])
def test_padded_planes_bit_identical(fm, alg, steps, unit, leaf, fused):
    m, k, n = (u * v for u, v in zip(unit, leaf))
    A, B, C0 = make_inputs(m, k, n, 77, "u11", np.float32, with_c=True)
    dev = lambda x: fm.col_major(torch.from_numpy(np.asfortranarray(x)).to(DEV))  # noqa: E731
    Ad, Bd = dev(A), dev(B)
    out = []
    for fusion in (1, 2):
        C = dev(C0)
        fm.fastmatmul(alg, Ad, Bd, C, steps, alpha=1.5, beta=-0.5, mode="split_bf16",
                      opts=fm.options(stage_fusion=fusion))
        out.append(C)
    torch.cuda.synchronize()
    assert torch.equal(out[0], out[1]), float((out[0] - out[1]).abs().max())
    prep = []
    try:
        for fusion in (1, 2):
            fm.set_stage_fusion(fusion)
            prep.append(fm.plan_info(alg, m, k, n, steps, dtype=torch.float32, mode="split_bf16")["prep_bytes"])
    finally:
        fm.set_stage_fusion(1)
    assert (prep[0] < prep[1]) == fused
