"""Population arrays of 4 GiB and more: the row kernel with scalar 64-bit
addresses (csrc/lbmib_fluid.hip, PtrRows) updates every cell to the same bits
as the vector-per-lane kernel, which addresses each cell by itself; walls,
inlet/outlet and periodic wrap on each axis, a ragged grid, one sheet."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bc", [(3, 1, 2), (1, 2, 1), (2, 1, 2)], ids=["ipw", "pwp", "wpw"])
def test_large_rows_match_the_general_addressing(bc):
    import lbmib
    kinds = {3: lbmib.BC_INOUT, 1: lbmib.BC_PERIODIC, 2: lbmib.BC_WALL}
    nx, ny, nz = 448, 255, 251
    assert 19 * nx * ny * nz * 8 >= 1 << 32  # where this form begins
    sheet = lbmib.Sheet.centred(20, 24, 1.0, (100.0, 120.0, 130.0), 1e-3, 1e-3, jitter=0.1, seed=3)
    out = []
    for shape in ((1, 3, 0), (1, 0, 0), (2, 1, 0)):
        print(f"large rows {bc} {shape}", flush=True)
        with lbmib.Engine(nx, ny, nz, bc=tuple(kinds[b] for b in bc), precision="f64", tau=0.7, rho0=1.0,
                          u0=(0.01, 0.0, 0.0), quirks=True, sheets=[sheet]) as e:
            e.set_kernel_variant(*shape)
            e.init()
            e.step(3)
            assert e.status() == 0
            out.append((e.df(), e.fibers(0)))
        if len(out) > 1:
            df, fib = out.pop()
            assert np.array_equal(df, out[0][0])
            assert np.array_equal(fib, out[0][1])
