"""The forward convolution's tile form (csrc/lbmib_surr.hip, k_conv_tile) at
the sizes where it changes: lines that do and do not fill a wave's positions,
tiles past the volume in y and z, input channels staged in slices, channel
groups past Cout, an odd number of reduction items per wave, several samples,
with bias, ReLU and mask; against oracle/surrogate_oracle.conv3d.

Tolerance: one rounding to BF16 of an FP32 sum, as in test_gpu_surrogate:
2^-8 (|ref| + a) + a with a = 2^-16 sum |terms|.
"""
import numpy as np
import pytest
import torch

from oracle import surrogate_oracle as so

pytestmark = pytest.mark.gpu


def _bf16(a):
    return torch.from_numpy(so.bf16_bits(a).view(np.int16)).to("cuda").view(torch.bfloat16)


def _host(t):
    torch.cuda.synchronize()
    return so.from_bf16_bits(t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16))


@pytest.mark.parametrize("case", [
    (1, 16, 16, 16, 64, 128),
    (1, 1, 1, 1, 64, 16),       # one voxel
    (2, 3, 2, 5, 32, 32),       # a whole sample in one wave
    (1, 8, 8, 8, 256, 128),     # narrow tiles, eight parts of the reduction
    (4, 8, 8, 8, 128, 256),
    (1, 13, 21, 27, 64, 96),    # 27 of 32 positions a line, partial tiles both ways, a partial channel group
    (2, 5, 7, 9, 256, 48),
    (1, 9, 10, 64, 64, 64),     # the longest lines
    (1, 7, 12, 63, 128, 80),    # all but the longest, channels in slices
    (1, 12, 14, 33, 256, 64),   # 33 of 64 positions, more slices
    (3, 20, 20, 20, 64, 256),
    (2, 32, 1, 16, 128, 128),   # one line a plane
    (2, 1, 40, 24, 128, 16),    # one plane a sample
    (4, 24, 32, 32, 64, 32),
    (1, 8, 8, 8, 32, 512),
], ids=lambda c: "x".join(map(str, c)))
def test_tile_matches_oracle(case):
    import surrogate as sg
    B, D, H, W, ci, co = case
    assert ci >= 64 or B * D * H * W < 4096  # where this form is taken
    print(f"conv tile {case}", flush=True)
    rng = np.random.default_rng(22)
    x = so.bf16_round(rng.standard_normal((B, D, H, W, ci)))
    w = so.bf16_round(rng.standard_normal((co, 27, ci)) / np.sqrt(27 * ci))
    b = rng.standard_normal(co).astype(np.float32).astype(np.float64) * 0.1
    m = so.bf16_round(np.maximum(rng.standard_normal((B, D, H, W, co)), 0.0))
    L = sg._bind()
    dx, dw, dm = _bf16(x), _bf16(w), _bf16(m)
    db = torch.from_numpy(b.astype(np.float32)).to("cuda")
    ref, plain = so.conv3d(x, w, b), so.conv3d(x, w)
    tot = so.conv3d(np.abs(x), np.abs(w), np.abs(b))
    a = 2.0 ** -16 * tot
    for relu, mask, want in ((0, None, ref), (1, None, np.maximum(ref, 0.0)), (0, dm, plain * (m > 0))):
        y = torch.full((B, D, H, W, co), 7.0, dtype=torch.bfloat16, device="cuda")
        sg.check(L.lbmib_sg_conv3d_fwd(sg.ptr(dx), sg.ptr(dw), None if mask is not None else sg.ptr(db), sg.ptr(mask),
                                       sg.ptr(y), B, D, H, W, ci, co, relu, sg.stream()), "conv fwd")
        bad = np.abs(_host(y) - want) > 2.0 ** -8 * (np.abs(want) + a) + a
        assert not bad.any(), (relu, mask is not None, int(bad.sum()))
