"""The forward convolution's forms (csrc/lbmib_surr.hip) where their shapes and
values are at an edge; against oracle/surrogate_oracle.conv3d.

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


def _conv(x, w, b, relu):
    import surrogate as sg
    L = sg._bind()
    B, D, H, W, ci = x.shape
    co = w.shape[0]
    dx, dw = _bf16(x), _bf16(w)
    db = None if b is None else torch.from_numpy(b.astype(np.float32)).to("cuda")
    y = torch.full((B, D, H, W, co), 7.0, dtype=torch.bfloat16, device="cuda")
    sg.check(L.lbmib_sg_conv3d_fwd(sg.ptr(dx), sg.ptr(dw), sg.ptr(db), None, sg.ptr(y), B, D, H, W, ci, co, relu,
                                   sg.stream()), "conv fwd")
    return _host(y)


@pytest.mark.parametrize("case", [
    (64, 1, 2048, 1, 64, 16),   # tiles of 512 lines of one plane
    (64, 2, 600, 1, 64, 32),    # of 256 lines of two planes
    (1, 3, 511, 1, 128, 48),
], ids=lambda c: "x".join(map(str, c)))
def test_lines_of_one_voxel(case):
    _against_oracle(case)


@pytest.mark.parametrize("case", [
    (600, 2, 2, 2, 64, 128),    # the general forms: many samples of few voxels
    (2500, 1, 1, 1, 256, 64),
    (70, 64, 1, 1, 64, 256),
    (1, 1700, 1, 16, 32, 48),   # one line a plane
    (200, 8, 8, 8, 16, 16),
    (40, 2, 2, 2, 64, 128),     # the tile: few samples of few voxels
], ids=lambda c: "x".join(map(str, c)))
def test_narrow_samples(case):
    _against_oracle(case)


def _against_oracle(case):
    B, D, H, W, ci, co = case
    print(f"conv edges {case}", flush=True)
    rng = np.random.default_rng(31)
    x = so.bf16_round(rng.standard_normal((B, D, H, W, ci)))
    w = so.bf16_round(rng.standard_normal((co, 27, ci)) / np.sqrt(27 * ci))
    b = rng.standard_normal(co).astype(np.float32).astype(np.float64) * 0.1
    ref = so.conv3d(x, w, b)
    a = 2.0 ** -16 * so.conv3d(np.abs(x), np.abs(w), np.abs(b))
    bad = np.abs(_conv(x, w, b, 0) - ref) > 2.0 ** -8 * (np.abs(ref) + a) + a
    assert not bad.any(), int(bad.sum())


def _with_infinities(case, relu):
    """x with +inf in one voxel's last channel and -inf in a far one's first: the outputs that read them are
    infinite (the weights hold no zero), and only those."""
    B, D, H, W, ci, co = case
    print(f"conv infinities {case}", flush=True)
    rng = np.random.default_rng(32)
    x = so.bf16_round(rng.standard_normal((B, D, H, W, ci)))
    w = so.bf16_round(rng.standard_normal((co, 27, ci)) / np.sqrt(27 * ci))
    assert (w != 0).all()
    x[0, D // 2, H // 2, W // 2, ci - 1] = np.inf
    if B > 1 or max(D, H, W) >= 8:
        x[B - 1, 0, 0, 0, 0] = -np.inf
    # the finite part, and the infinite voxels' products on top of it (which the oracle's zero padding does not meet)
    fin = np.where(np.isfinite(x), x, 0.0)
    ref = so.conv3d(fin, w)
    a = 2.0 ** -16 * so.conv3d(np.abs(fin), np.abs(w))
    for b, z, y, xx, c in np.argwhere(np.isinf(x)):
        for dz in (-1, 0, 1):
            for dy in (-1, 0, 1):
                for dx in (-1, 0, 1):
                    p = (z - dz, y - dy, xx - dx)
                    if all(0 <= v < n for v, n in zip(p, (D, H, W))):
                        ref[(b,) + p] += x[b, z, y, xx, c] * w[:, 9 * (dz + 1) + 3 * (dy + 1) + dx + 1, c]
    if relu:
        ref = np.maximum(ref, 0.0)
    got = _conv(x, w, None, relu)
    inf = np.isinf(ref)
    assert inf.any() and not np.isnan(ref).any()
    np.testing.assert_array_equal(got[inf], ref[inf])
    got, ref, a = got[~inf], ref[~inf], a[~inf]
    assert np.isfinite(got).all()
    bad = np.abs(got - ref) > 2.0 ** -8 * (np.abs(ref) + a) + a
    assert not bad.any(), int(bad.sum())


@pytest.mark.parametrize("relu", [0, 1])
@pytest.mark.parametrize("case", [
    (1, 16, 16, 16, 64, 128),
    (1, 8, 8, 8, 256, 128),     # eight parts of the reduction
    (1, 13, 21, 27, 64, 96),
    (2, 5, 7, 9, 256, 48),
    (1, 12, 14, 33, 256, 64),   # channels in slices
    (4, 24, 32, 32, 64, 32),
    (1, 8, 8, 8, 32, 512),
    (1, 1, 1, 1, 64, 16),
], ids=lambda c: "x".join(map(str, c)))
def test_tile_keeps_an_infinity(case, relu):
    _with_infinities(case, relu)


@pytest.mark.parametrize("relu", [0, 1])
@pytest.mark.parametrize("case", [
    (2, 12, 33, 33, 16, 32),
    (3, 7, 40, 31, 16, 16),
    (1, 8, 64, 64, 16, 48),
    (1, 6, 64, 64, 32, 32),
], ids=lambda c: "x".join(map(str, c)))
def test_march_keeps_an_infinity(case, relu):
    _with_infinities(case, relu)


def test_more_samples_than_a_launch_has_blocks():
    """8.4 million samples of one voxel: each output is the centre tap's product."""
    import surrogate as sg
    B, ci, co = (1 << 23) + 16, 64, 16
    print(f"conv samples {B}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(33)
    x = torch.randn((B, ci), generator=gen, device="cuda", dtype=torch.bfloat16)
    w = (torch.randn((co, 27, ci), generator=gen, device="cuda") / 8).to(torch.bfloat16)
    y = torch.full((B, co), 7.0, dtype=torch.bfloat16, device="cuda")
    sg.check(sg._bind().lbmib_sg_conv3d_fwd(sg.ptr(x), sg.ptr(w), None, None, sg.ptr(y), B, 1, 1, 1, ci, co, 0,
                                            sg.stream()), "conv fwd")
    torch.cuda.synchronize()
    wc = w[:, 13].double()
    for b in (0, B // 2 - 100000, B - 100000):
        xs = x[b:b + 100000].double()
        ref, a = xs @ wc.T, 2.0 ** -16 * (xs.abs() @ wc.abs().T)
        bad = (y[b:b + 100000].double() - ref).abs() > 2.0 ** -8 * (ref.abs() + a) + a
        assert not bad.any(), (b, int(bad.sum()))
