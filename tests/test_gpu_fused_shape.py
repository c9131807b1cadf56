"""The automatic shape of the fused launch: sizes on both sides of each line
of its rule (rows of whole 64-byte pieces or not, rows of one cache line,
arrays within the Infinity Cache or not, x pairs, wall and periodic x) give
the bits of one cell per lane with nontemporal accesses, batches too."""
import numpy as np
import pytest

import lbmib

pytestmark = pytest.mark.gpu

IPW = (lbmib.BC_INOUT, lbmib.BC_PERIODIC, lbmib.BC_WALL)
WPW = (lbmib.BC_WALL, lbmib.BC_PERIODIC, lbmib.BC_WALL)
PPW = (lbmib.BC_PERIODIC, lbmib.BC_PERIODIC, lbmib.BC_WALL)


def _args(prec, nx, ny, nz, bc=IPW):
    sheet = lbmib.Sheet.centred(9, 9, 1.0, (nx / 3.0, ny / 2.0, nz / 2.0), 2e-3, 2e-3, jitter=0.1, seed=3)
    return dict(nx=nx, ny=ny, nz=nz, bc=bc, tau=0.7, rho0=1.0, u0=(0.02, 0.0, 0.0), quirks=True, sheets=[sheet],
                precision=prec)


def _state(e):
    return [e.df(), e.fibers(0)]


CASES = [
    ("f16", 64, 24, 20, IPW), ("f16", 50, 24, 20, IPW), ("f16", 128, 200, 200, IPW), ("f16", 272, 20, 20, IPW),
    ("bf16", 300, 20, 20, WPW), ("f32", 32, 20, 24, IPW), ("f32", 97, 20, 24, IPW), ("f32", 96, 160, 160, IPW),
    ("f32", 50, 200, 200, IPW), ("f32", 128, 140, 140, PPW), ("f64", 24, 20, 24, IPW), ("f64", 128, 100, 100, IPW),
    ("f64", 60, 150, 150, IPW), ("f64", 101, 40, 30, WPW),
]


@pytest.mark.parametrize("prec,nx,ny,nz,bc", CASES)
def test_automatic_shape_same_bits(prec, nx, ny, nz, bc):
    out = []
    for variant in ((0, -1, 0), (1, 3, 0)):
        with lbmib.Engine(**_args(prec, nx, ny, nz, bc)) as e:
            e.set_kernel_variant(*variant)
            e.init()
            e.step(5)
            assert e.status() == 0
            out.append(_state(e))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("prec,edge", [("f32", 100), ("f64", 50), ("f16", 50)])
def test_batch_same_bits(prec, edge):
    kw = [_args(prec, edge, 40, 36), _args(prec, 64, 24, 24)]
    with lbmib.Batch(kw) as b:
        b.init()
        b.step(4)
        got = [_state(e) for e in b.instances]
    for k, g in zip(kw, got):
        with lbmib.Engine(**k) as e:
            e.init()
            e.step(4)
            for a, c in zip(_state(e), g):
                assert np.array_equal(a, c)
