"""The weight gradient (csrc/lbmib_surr.hip, k_conv_wgrad) on lines so long that
a unit's byte offsets pass 2^31, with output channels that are no multiple of
32: few voxels set, the reference over those in FP64.

Tolerance: FP32 sums of exact BF16 products, |gpu - ref| <= 2^-18 sum |terms|.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("co", [48, 32])
def test_long_lines(co):
    import surrogate as sg
    W, ci = (1 << 21) - 3, 256
    assert 3 * W * ci * 2 >= 1 << 31
    print(f"wgrad long lines {W} {ci} {co}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(41)
    x = torch.zeros((W, ci), dtype=torch.bfloat16, device="cuda")
    dy = torch.zeros((W, co), dtype=torch.bfloat16, device="cuda")
    at = torch.randint(1, W - 1, (500,), generator=gen, device="cuda")
    at[:4] = torch.tensor([0, 1, W - 2, W - 1], device="cuda")
    at = torch.unique(at)
    dy[at] = torch.randn((len(at), co), generator=gen, device="cuda").to(torch.bfloat16)
    for o in (-1, 0, 1):
        x[(at + o).clamp(0, W - 1)] = torch.randn((len(at), ci), generator=gen, device="cuda").to(torch.bfloat16)
    dw = torch.full((co, 27, ci), 7.0, dtype=torch.float32, device="cuda")
    db = torch.full((co,), 7.0, dtype=torch.float32, device="cuda")
    sg.check(sg._bind().lbmib_sg_conv3d_bwd_weight(sg.ptr(x), sg.ptr(dy), sg.ptr(dw), sg.ptr(db), 1, 1, 1, W, ci, co,
                                                   sg.stream()), "conv bwd weight")
    torch.cuda.synchronize()
    g = dy[at].double().cpu().numpy()
    rw, aw = np.zeros((co, 27, ci)), np.zeros((co, 27, ci))
    for ox in (-1, 0, 1):
        v = at + ox
        xs = x[v.clamp(0, W - 1)].double().cpu().numpy()
        xs[((v < 0) | (v >= W)).cpu().numpy()] = 0.0
        rw[:, 13 + ox] = g.T @ xs
        aw[:, 13 + ox] = np.abs(g).T @ np.abs(xs)
    assert np.all(np.abs(dw.cpu().numpy() - rw) <= 2.0 ** -18 * aw + 1e-30)
    assert np.all(np.abs(db.cpu().numpy() - g.sum(0)) <= 2.0 ** -18 * np.abs(g).sum(0) + 1e-30)
