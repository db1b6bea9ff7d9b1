"""A uniform flow is a solution that every scheme here keeps: all faces of an axis have the same flux, and the
residual is made of their differences.  In the FP32-residual form the increments that are added to the
double state are then exact zeros, so the state stays bitwise as it is, on sizes whose cell sizes no
float holds exactly, at and beside the 60 columns of a wavefront."""
import numpy as np
import pytest

from turbostructred_amd import capi
import util

pytestmark = pytest.mark.gpu

VELOCITY = (0.37, -0.81, 0.23)
FLOWS = [(0.5323, 0.3), (0.138, 0.029), (1.1, 70.0)]  # density, pressure: about Mach 1, 2 and 0.1


def after_steps(n, riemann, recon, stages, periodic, rho, p, velocity=VELOCITY):
    nd = len(n)
    shape = dict(zip(("nx", "ny", "nz"), n))
    cfg = capi.make_config(ndims=nd, ly=0.7, lz=0.9, cfl=0.4, riemann=riemann, recon=recon, rk_stages=stages,
                           precision=capi.FP32_RESIDUAL, eps=0.05, periodic=(periodic,) * nd + (0,) * (3 - nd),
                           bcs=[dict(type=capi.BC_NATURAL)], **shape)
    vel = velocity[:nd] + (0.0,) * (3 - nd)
    U = util.fill_state(cfg, lambda x, y, z: util.prim2cons(rho + 0 * x, *vel, p, cfg.gamma))
    U = U.astype(np.float32).astype(np.float64)  # forward Euler adds to the float form of the state
    s = capi.Solver(cfg)
    s.set_state(U)
    info = s.step(20)
    got = capi.interior(cfg, s.get_state())
    s.close()
    assert info.steps_done == 20
    return got, capi.interior(cfg, U)


@pytest.mark.parametrize("rho,p", FLOWS)
@pytest.mark.parametrize("periodic", [0, 1])
@pytest.mark.parametrize("recon", [capi.RECON_PWC, capi.RECON_LINEAR_LIM])
@pytest.mark.parametrize("riemann", [capi.RIEMANN_ROE, capi.RIEMANN_HLLC])
@pytest.mark.parametrize("stages", [1, 3])
@pytest.mark.parametrize("n", [(59,), (60,), (61,), (203,), (61, 7), (130, 21)])
def test_lines_and_planes(n, stages, riemann, recon, periodic, rho, p):
    got, ref = after_steps(n, riemann, recon, stages, periodic, rho, p)
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("rho,p", FLOWS)
@pytest.mark.parametrize("periodic", [0, 1])
@pytest.mark.parametrize("recon", [capi.RECON_PWC, capi.RECON_LINEAR_LIM])
@pytest.mark.parametrize("riemann", [capi.RIEMANN_ROE, capi.RIEMANN_HLLC])
@pytest.mark.parametrize("stages", [1, 3])
@pytest.mark.parametrize("n", [(5, 3, 4), (61, 7, 15), (33, 21, 29)])
def test_boxes(n, stages, riemann, recon, periodic, rho, p):
    got, ref = after_steps(n, riemann, recon, stages, periodic, rho, p)
    assert np.array_equal(got, ref)
