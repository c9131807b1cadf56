"""The weight gradient (csrc/lbmib_surr.hip) of volumes whose lines are one
voxel, which it takes along another axis (wgrad_view); against
oracle/surrogate_oracle.conv3d_bwd_weight.

Tolerance: FP32 sums of exact BF16 products, |gpu - ref| <= 2^-18 sum |terms|.
"""
import numpy as np
import pytest
import torch

from oracle import surrogate_oracle as so

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", [
    (64, 1, 1, 1, 32, 48),     # samples of one voxel: lines of 64
    (97, 1, 1, 1, 32, 32),     # no line length divides them
    (1, 1, 1, 1, 16, 32),
    (500, 1, 1, 1, 256, 16),
    (3, 1, 70, 1, 32, 32),     # lines along y, longer than 64
    (2, 5, 33, 1, 64, 80),
    (3, 70, 1, 1, 32, 16),     # lines along z
    (40, 7, 1, 1, 16, 16),
], ids=lambda c: "x".join(map(str, c)))
def test_lines_of_one_voxel(case):
    import surrogate as sg
    B, D, H, W, ci, co = case
    print(f"wgrad narrow {case}", flush=True)
    rng = np.random.default_rng(51)
    x = so.bf16_round(rng.standard_normal((B, D, H, W, ci)))
    dy = so.bf16_round(rng.standard_normal((B, D, H, W, co)))
    dx, dd = (torch.from_numpy(so.bf16_bits(a).view(np.int16)).to("cuda").view(torch.bfloat16) for a in (x, dy))
    dw = torch.full((co, 27, ci), 7.0, dtype=torch.float32, device="cuda")
    db = torch.full((co,), 7.0, dtype=torch.float32, device="cuda")
    sg.check(sg._bind().lbmib_sg_conv3d_bwd_weight(sg.ptr(dx), sg.ptr(dd), sg.ptr(dw), sg.ptr(db), B, D, H, W, ci, co,
                                                   sg.stream()), "conv bwd weight")
    torch.cuda.synchronize()
    rw, rb = so.conv3d_bwd_weight(x, dy)
    aw, ab = so.conv3d_bwd_weight(np.abs(x), np.abs(dy))
    assert np.all(np.abs(dw.cpu().numpy() - rw) <= 2.0 ** -18 * aw + 1e-30)
    assert np.all(np.abs(db.cpu().numpy() - rb) <= 2.0 ** -18 * ab + 1e-30)


def test_a_neighbouring_samples_infinity_stays_out():
    import surrogate as sg
    B, ci, co = 64, 16, 16
    x = torch.ones((B, ci), dtype=torch.bfloat16, device="cuda")
    dy = torch.ones((B, co), dtype=torch.bfloat16, device="cuda")
    x[5, 3] = float("inf")
    dw = torch.full((co, 27, ci), 7.0, dtype=torch.float32, device="cuda")
    sg.check(sg._bind().lbmib_sg_conv3d_bwd_weight(sg.ptr(x), sg.ptr(dy), sg.ptr(dw), None, B, 1, 1, 1, ci, co,
                                                   sg.stream()), "conv bwd weight")
    torch.cuda.synchronize()
    want = torch.zeros((co, 27, ci))
    want[:, 13] = B
    want[:, 13, 3] = float("inf")
    assert torch.equal(dw.cpu(), want)
