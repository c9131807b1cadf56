"""The forward convolution's marching form (csrc/lbmib_surr.hip, k_conv_march)
at the sizes where it changes: lines that do and do not fill a wave's 64 or
48 positions, line groups past the plane's end, one plane, channel tiles past
Cout, with bias, ReLU and mask; against oracle/surrogate_oracle.conv3d.

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
    (1, 6, 64, 64, 32, 32),    # a line a wave
    (2, 12, 33, 33, 16, 32),   # 33 of 48 positions, a partial line group
    (1, 13, 43, 48, 32, 48),   # 48 positions, a half channel tile
    (1, 9, 57, 50, 32, 16),
    (3, 7, 40, 31, 16, 16),    # two lines a wave, the second ending inside a fragment
    (24, 1, 64, 16, 32, 64),   # one plane a sample, several channel tiles
    (1, 45, 36, 17, 32, 32),
    (6, 16, 32, 9, 16, 48),
], ids=lambda c: "x".join(map(str, c)))
def test_march_matches_oracle(case):
    import surrogate as sg
    B, D, H, W, ci, co = case
    assert B * D * H * W >= 24576  # where this form begins
    print(f"conv march {case}", flush=True)
    rng = np.random.default_rng(21)
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
