"""Fiber forces, spreading and move against the FP64 oracle where the kernels'
tiles can go wrong: node counts around a wave, sheets that share a wave, tiles
with few and many candidates, sheets one behind the other in the same (y, z)
bins, a support box wider than a tile's lanes, dense sheets.

Tolerance: both sides sum the same FP64 terms in the same order, up to the
device's cosine (2 units of the last place) and contraction in the spread sum
(64 terms), over the steps taken: 64 * 2.2e-16 * 16 steps < 1e-12, times 10.
"""
import numpy as np
import pytest

import lbmib
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

TOL = 1e-11
N = (48, 44, 40)
BC = (lbmib.BC_INOUT, lbmib.BC_PERIODIC, lbmib.BC_WALL)


def _sheet(rows, cols, spacing, x, y=None, z=None, lean=0.0, jitter=0.2, seed=1):
    """A sheet around (x, y, z); lean tilts it so that its x range grows."""
    w, h = spacing * (cols - 1), spacing * (rows - 1)
    y = N[1] / 2.0 if y is None else y
    z = N[2] / 2.0 if z is None else z
    xyz = lbmib.sheet_positions(rows, cols, w, h, x, y - h / 2, z - w / 2)
    xyz[..., 0] += lean * (xyz[..., 1] - y)
    xyz += np.random.default_rng(seed).uniform(-jitter * spacing, jitter * spacing, xyz.shape)
    return lbmib.Sheet(rows, cols, w, h, 1e-3, 1e-3, xyz)


CASES = {
    "one_wave": [_sheet(8, 8, 1.0, 20.0)],
    "one_more_than_a_wave": [_sheet(5, 13, 1.0, 20.0)],
    "one_less": [_sheet(7, 9, 1.0, 20.0)],
    "sheets_in_one_wave": [_sheet(4, 5, 1.0, 14.0, y=14.0, seed=1), _sheet(4, 4, 1.0, 20.0, z=26.0, seed=2),
                           _sheet(5, 4, 1.0, 26.0, y=28.0, seed=3), _sheet(6, 11, 1.0, 32.0, seed=4)],
    "behind_each_other": [_sheet(20, 21, 1.0, 18.0, seed=5), _sheet(20, 21, 1.0, 20.5, seed=6),
                          _sheet(20, 21, 1.0, 30.0, seed=7)],
    "six_behind_each_other": [_sheet(14, 15, 1.0, 9.0 + 5.0 * k, seed=8 + k) for k in range(6)],
    "six_close": [_sheet(14, 15, 1.0, 14.0 + 2.0 * k, seed=20 + k) for k in range(6)],
    "leaning": [_sheet(21, 18, 1.0, 23.0, lean=0.9)],
    "dense": [_sheet(24, 25, 0.55, 20.0)],
    "very_dense": [_sheet(30, 30, 0.45, 20.0)],
    "coarse": [_sheet(9, 8, 2.7, 20.0)],
}


@pytest.mark.parametrize("name", CASES)
def test_against_oracle(name):
    sheets, u0, steps = CASES[name], (0.02, 0.0, 0.0), 16
    o = Oracle(*N, BC, 0.7, 1.0, u0, True)
    for s in sheets:
        o.add_sheet(s.rows, s.cols, s.width, s.height, s.ks, s.kb, s.xyz)
    o.init()
    o.preshift(all_sheets=True)
    assert o.step(steps) == 0
    with lbmib.Engine(*N, bc=BC, precision="f64", tau=0.7, rho0=1.0, u0=u0, quirks=True, sheets=sheets) as e:
        e.init()
        e.step(steps)
        assert e.status() == 0
        _, vel = e.macroscopic()
        assert np.abs(vel - o.vel()).max() <= TOL * np.abs(o.vel()).max()
        for k, s in enumerate(sheets):
            got, want = e.fibers(k), o.nodes(k)
            assert np.abs(got[..., :3] - want[..., :3]).max() <= TOL * max(N)
