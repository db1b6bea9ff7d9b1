"""3-D stages around the number of planes a workgroup outputs (6 in double; 14, and 10 in stage 2, in
the FP32-residual form) and the 60 columns of a strip: whole blocks, one plane over and one short, fewer
planes than one block, open and periodic, against the oracle."""
import numpy as np
import pytest

from turbostructred_amd import capi
from oracle import pyoracle
import util

pytestmark = pytest.mark.gpu

# FP32 residual: float rounding (6e-8) of the face states and fluxes, a few per step of at most
# CFL 0.4 of the state: below 1e-6 after 4 steps
TOL = {capi.FP64: 1e-12, capi.FP32_RESIDUAL: 2e-6}


@pytest.mark.parametrize("precision", [capi.FP64, capi.FP32_RESIDUAL])
@pytest.mark.parametrize("periodic", [0, 1])
@pytest.mark.parametrize("shape", [(60, 5, 2), (61, 4, 5), (7, 9, 6), (62, 3, 7), (5, 6, 10), (9, 4, 11), (60, 5, 13), (4, 7, 14),
                                   (59, 2, 15), (6, 5, 29)])
def test_planes(shape, periodic, precision):
    nx, ny, nz = shape
    cfg = capi.make_config(ndims=3, nx=nx, ny=ny, nz=nz, cfl=0.4, riemann=capi.RIEMANN_HLLC, recon=capi.RECON_LINEAR_LIM,
                           rk_stages=3, precision=precision, periodic=(periodic,) * 3,
                           bcs=[dict(type=capi.BC_NATURAL), dict(type=capi.BC_WALL), dict(type=capi.BC_SYMMETRY)],
                           side_marker=(0, 1, 2, 0, 1, 2))

    def wave(x, y, z):
        rho = 1 + 0.2 * np.sin(2 * np.pi * x) * np.cos(2 * np.pi * y) + 0.1 * np.cos(2 * np.pi * z)
        return util.prim2cons(rho, 0.3 * np.cos(2 * np.pi * y), 0.2 * np.sin(2 * np.pi * z), -0.2 * np.sin(2 * np.pi * x),
                              1 + 0.1 * np.cos(2 * np.pi * (x - z)), cfg.gamma)

    U = util.fill_state(cfg, wave)
    s = capi.Solver(cfg)
    s.set_state(U)
    info = s.step(4)
    a = capi.interior(cfg, s.get_state())
    s.close()
    cfg.precision = capi.FP64
    o = pyoracle.Oracle(cfg)
    o.set_state(U)
    ref = o.step(4)
    assert abs(info.time - ref.time) <= TOL[precision] * ref.time
    assert util.normwise_rel(a, capi.interior(cfg, o.get_state())).max() <= TOL[precision]
