"""Lists of layers in one launch (transposed weights, Adam), the wide MSE and
the pooling kernels at the edges of their tiles and vectors."""
import pytest
import torch

import surrogate as sg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chans", [[(16, 16)], [(48, 32), (16, 256), (272, 64), (64, 64)], [(16, 16)] * 35])
@pytest.mark.parametrize("shift", [0, 1])
def test_flip_many(chans, shift):
    """wt[ci][26 - t][co] = w[co][t][ci], copied bits, also from pointers off 16 bytes."""
    L, g = sg._bind(), torch.Generator(device="cuda").manual_seed(3)
    ws, wts = [], []
    items = (sg.FlipItem * len(chans))()
    for k, (ci, co) in enumerate(chans):
        n = co * 27 * ci
        ws.append(torch.randn(n + 8, generator=g, device="cuda").to(torch.bfloat16)[shift:shift + n])
        wts.append(torch.zeros(n + 8, dtype=torch.bfloat16, device="cuda"))
        items[k] = sg.FlipItem(ws[k].data_ptr(), wts[k].data_ptr(), ci, co)
    sg.check(L.lbmib_sg_flip_many(len(chans), items, sg.stream()), "flip")
    for (ci, co), w, wt in zip(chans, ws, wts):
        want = w.view(co, 27, ci).permute(2, 1, 0).flip(1)
        assert torch.equal(wt[:co * 27 * ci].view(ci, 27, co), want)
        assert not wt[co * 27 * ci:].any()


def test_flip_many_refuses():
    L, t = sg._bind(), torch.zeros(16 * 27 * 16, dtype=torch.bfloat16, device="cuda")
    for ci, co in ((16, 24), (8, 16), (20, 16), (16, 512)):
        items = (sg.FlipItem * 1)(sg.FlipItem(t.data_ptr(), t.data_ptr(), ci, co))
        assert L.lbmib_sg_flip_many(1, items, sg.stream()) != 0


@pytest.mark.parametrize("sizes", [[1], [3, 4, 5, 1023, 1024, 1025, 70001], [16] * 33, [4096, 7] * 40])
@pytest.mark.parametrize("shift", [0, 1])
def test_adam_many_is_adam(sizes, shift):
    """One launch over a list gives the bits of a call per tensor."""
    L = sg._bind()
    outs = []
    for many in (False, True):
        g = torch.Generator(device="cuda").manual_seed(9)
        new = lambda n: torch.randn(n + 1, generator=g, device="cuda")[shift:shift + n]  # noqa: E731
        ts = [[new(n), new(n), new(n), new(n).abs(), torch.zeros(n + 1, dtype=torch.bfloat16, device="cuda")[shift:shift + n]]
              for n in sizes]
        if many:
            items = (sg.AdamItem * len(ts))()
            for k, t in enumerate(ts):
                items[k] = sg.AdamItem(*(x.data_ptr() for x in t[:4]), t[4].data_ptr() if k % 3 else None, t[0].numel())
            sg.check(L.lbmib_sg_adam_many(len(ts), items, 1e-3, 0.9, 0.999, 1e-8, 3, sg.stream()), "adam")
        else:
            for k, t in enumerate(ts):
                sg.check(L.lbmib_sg_adam(*(sg.ptr(x) for x in t[:4]), sg.ptr(t[4]) if k % 3 else None, t[0].numel(), 1e-3,
                                         0.9, 0.999, 1e-8, 3, sg.stream()), "adam")
        outs.append(ts)
    for k, (a, b) in enumerate(zip(*outs)):
        for x, y in zip(a, b):
            assert torch.equal(x, y)
        assert (k % 3 == 0) == (not a[4].any())


@pytest.mark.parametrize("M,C,nl", [(1, 16, 4), (777, 16, 4), (1000, 8, 8), (333, 24, 11), (500, 12, 4), (70000, 16, 16)])
def test_mse(M, C, nl):
    """Gradient 2 (out - tgt) / (M nl) rounded once to BF16 (relative 2^-8); the
    loss a sum of M nl squares in FP32, 256 x 1024 partial sums: within
    (terms per lane + 20) * 2^-24 of the 64-bit sum, here 1e-5."""
    L, g = sg._bind(), torch.Generator(device="cuda").manual_seed(5)
    out = torch.randn((M, C), generator=g, device="cuda").to(torch.bfloat16)
    tgt = torch.randn((M, nl), generator=g, device="cuda")
    dout, loss = torch.full_like(out, 7.0), torch.zeros(1, device="cuda")
    sg.check(L.lbmib_sg_mse(sg.ptr(out), sg.ptr(tgt), sg.ptr(dout), sg.ptr(loss), M, C, nl, sg.stream()), "mse")
    d = out[:, :nl].double() - tgt.double()
    want = 2.0 * d / (M * nl)
    assert abs(loss.item() - (d * d).mean().item()) <= 1e-5 * (d * d).mean().item()
    assert ((dout[:, :nl].double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-30).all()
    assert not dout[:, nl:].any()
