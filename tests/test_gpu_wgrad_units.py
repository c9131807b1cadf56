"""The weight gradient's units (csrc/lbmib_surr.hip, k_conv_wgrad) at the
sizes where they change: lines that are not whole runs of 8, lines longer than
a segment, planes packed into one unit across samples, partial line groups,
offsets past 32 bits; against oracle/surrogate_oracle.conv3d_bwd_weight.

Tolerance: FP32 sums of exact BF16 products, |gpu - ref| <= 2^-18 sum |terms|
(under 64 roundings of 2^-24 along any chain of partial sums).
"""
import numpy as np
import pytest
import torch

from oracle import surrogate_oracle as so

pytestmark = pytest.mark.gpu


def _bf16(a):
    return torch.from_numpy(so.bf16_bits(a).view(np.int16)).to("cuda").view(torch.bfloat16)


def _wgrad(x, dy, shape, ci, co):
    import surrogate as sg
    L = sg._bind()
    dw = torch.full((co, 27, ci), 7.0, dtype=torch.float32, device="cuda")
    db = torch.full((co,), 7.0, dtype=torch.float32, device="cuda")
    sg.check(L.lbmib_sg_conv3d_bwd_weight(sg.ptr(x), sg.ptr(dy), sg.ptr(dw), sg.ptr(db), *shape, ci, co, sg.stream()),
             "conv bwd weight")
    torch.cuda.synchronize()
    return dw.cpu().numpy().astype(np.float64), db.cpu().numpy().astype(np.float64)


@pytest.mark.parametrize("case", [
    (3, 5, 1, 1, 32, 32),     # one voxel a plane: planes of several samples in a unit
    (2, 3, 7, 5, 16, 32),     # a run of 8 not full, two planes a unit
    (1, 4, 5, 33, 32, 16),    # a fifth run of one voxel, a partial line group
    (1, 2, 3, 64, 32, 48),    # the longest whole line, a partial line group, a half channel tile
    (1, 2, 2, 65, 32, 32),    # segments, the last of one voxel
    (2, 1, 9, 100, 16, 16),   # segments and partial line groups, one plane a sample
    (1, 3, 10, 48, 64, 80),
    (5, 1, 4, 4, 256, 32),
], ids=lambda c: "x".join(map(str, c)))
def test_weight_gradient_units(case):
    B, D, H, W, ci, co = case
    print(f"wgrad units {case}", flush=True)
    rng = np.random.default_rng(11)
    x = so.bf16_round(rng.standard_normal((B, D, H, W, ci)))
    dy = so.bf16_round(rng.standard_normal((B, D, H, W, co)))
    dw, db = _wgrad(_bf16(x), _bf16(dy), (B, D, H, W), ci, co)
    rw, rb = so.conv3d_bwd_weight(x, dy)
    aw, ab = so.conv3d_bwd_weight(np.abs(x), np.abs(dy))
    assert np.all(np.abs(dw - rw) <= 2.0 ** -18 * aw + 1e-30)
    assert np.all(np.abs(db - rb) <= 2.0 ** -18 * ab + 1e-30)


@pytest.mark.parametrize("W", [5, 33, 65])
def test_an_infinity_stays_with_its_own_taps(W):
    """x infinite at the end of a line: the taps that no voxel reads it through stay finite."""
    B, D, H, ci, co = 1, 3, 6, 32, 32
    rng = np.random.default_rng(12)
    x = so.bf16_round(rng.standard_normal((B, D, H, W, ci)))
    dy = so.bf16_round(1.0 + rng.random((B, D, H, W, co)))  # no zeros: infinity times dy is infinity
    x[0, 1, H - 1, W - 1, 3] = np.inf
    dw, db = _wgrad(_bf16(x), _bf16(dy), (B, D, H, W), ci, co)
    with np.errstate(invalid="ignore"):
        rw, _ = so.conv3d_bwd_weight(x, dy)
    fin = np.isfinite(rw)
    assert not fin.all()
    np.testing.assert_array_equal(np.isfinite(dw), fin)
    np.testing.assert_array_equal(dw[~fin], rw[~fin])
    assert np.isfinite(db).all()


def test_offsets_past_32_bits():
    """Lines so long that a unit's byte offsets pass 2^31: few voxels set, the reference over those."""
    W, ci, co = 1 << 21, 256, 16
    shape = (1, 1, 2, W)
    gen = torch.Generator(device="cuda").manual_seed(13)
    x = torch.zeros((2, W, ci), dtype=torch.bfloat16, device="cuda")
    dy = torch.zeros((2, W, co), dtype=torch.bfloat16, device="cuda")
    at = torch.randint(1, W - 1, (600,), generator=gen, device="cuda")
    at[:4] = torch.tensor([0, 1, W - 2, W - 1], device="cuda")
    for y in range(2):
        dy[y, at] = torch.randn((len(at), co), generator=gen, device="cuda").to(torch.bfloat16)
        for o in (-1, 0, 1):
            v = (at + o).clamp(0, W - 1)
            x[y, v] = torch.randn((len(at), ci), generator=gen, device="cuda").to(torch.bfloat16)
    dw, db = _wgrad(x, dy, shape, ci, co)
    rw, aw = np.zeros((co, 27, ci)), np.zeros((co, 27, ci))
    at = torch.unique(at)
    for y in range(2):
        g = dy[y, at].double().cpu().numpy()
        for oy in (-1, 0, 1):
            for ox in (-1, 0, 1):
                if not 0 <= y + oy < 2:
                    continue
                v = at + ox
                xs = x[y + oy, v.clamp(0, W - 1)].double().cpu().numpy()
                xs[((v < 0) | (v >= W)).cpu().numpy()] = 0.0
                t = 9 + 3 * (oy + 1) + ox + 1
                rw[:, t] += g.T @ xs
                aw[:, t] += np.abs(g).T @ np.abs(xs)
    assert np.all(np.abs(dw - rw) <= 2.0 ** -18 * aw + 1e-30)
    gd = dy.double().cpu().numpy().reshape(-1, co)
    assert np.all(np.abs(db - gd.sum(0)) <= 2.0 ** -18 * np.abs(gd).sum(0) + 1e-30)
