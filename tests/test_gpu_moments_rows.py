"""The read of every cell's moments by rows: each storage form, boundary kind of
the axes, first step and later ones, with the force of a sheet at an edge.

The stored values are FP32; against the FP64 fields of the same state they are
off by their own rounding (2^-24 relative) and, in the deviation forms, by a sum
of 19 FP32 terms below 1 (19 * 2^-24 < 1.2e-6)."""
import numpy as np
import pytest
import torch

import lbmib

pytestmark = pytest.mark.gpu

B = {"i": lbmib.BC_INOUT, "p": lbmib.BC_PERIODIC, "w": lbmib.BC_WALL}


@pytest.mark.parametrize("prec", ["f64", "f32", "f16", "bf16"])
@pytest.mark.parametrize("nx,bc", [(64, "ipw"), (128, "wpw"), (192, "ppp"), (64, "iww")])
def test_rows_moments(prec, nx, bc):
    xyz = lbmib.sheet_positions(8, 9, 8.0, 7.0, nx - 9.3, 3.4, 4.2)
    with lbmib.Engine(nx, 24, 20, bc=tuple(B[c] for c in bc), precision=prec, tau=0.6, rho0=1.0, u0=(0.04, 0.0, 0.0),
                      quirks=True, g=1e-6, sheets=[lbmib.Sheet(8, 9, 8.0, 7.0, 3e-3, 3e-3, xyz)]) as e:
        e.init()
        out = torch.empty((4, 20, 24, nx), device="cuda")
        for steps in (0, 1, 4):
            e.step(steps)
            out.fill_(7.0)
            torch.cuda.synchronize()
            e.coarse_moments(1, out.data_ptr())
            e.sync()
            rho, vel = e.macroscopic()
            tol = 1.2e-7 if prec == "f64" else 1.3e-6
            assert np.abs(out[0].cpu().numpy() - rho).max() <= tol
            assert np.abs(out[1:].cpu().numpy() - vel).max() <= tol
