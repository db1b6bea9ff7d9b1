"""2-D viscous fluxes formed in the stage kernels: grids at and beside the 60 columns of a wavefront and
with few rows, every pairing of periodic and bounded axes, stretched cells, with and without momentum
out of the plane (the kernels for plane flows carry four variables), one and three stages, against
the oracle; and a plane flow against the same flow with a whisper of out-of-plane momentum."""
import numpy as np
import pytest

from turbostructred_amd import capi
from oracle import pyoracle
import util

pytestmark = pytest.mark.gpu

BCS = [dict(type=capi.BC_WALL), dict(type=capi.BC_MOVING_WALL, velocity=(0.3, 0.1, 0.0)), dict(type=capi.BC_SYMMETRY),
       dict(type=capi.BC_NATURAL)]


def config(nx, ny, periodic, stages, **kw):
    xy = [util.stretched(n, length, 1.0 + 1.0 / n) if n % 2 == 0 else (None, None) for n, length in ((nx, 1.0), (ny, 0.7))]
    xy = [xy[0] if not periodic[0] else (None, None), xy[1] if not periodic[1] else (None, None)]
    return capi.make_config(ndims=2, nx=nx, ny=ny, ly=0.7, cfl=0.4, riemann=capi.RIEMANN_ROE, eps=0.05,
                            recon=capi.RECON_LINEAR_LIM, rk_stages=stages, periodic=(*periodic, 0), bcs=BCS,
                            side_marker=(0, 3, 1, 2, 0, 0), viscous=True, viscosity=0.02, sigma=(0.4, -0.2, 0.0),
                            accel=(0.0, -0.3, 0.0), coord=[xy[0][0], xy[1][0], None], h=[xy[0][1], xy[1][1], None], **kw)


def flow(cfg, w):
    def f(x, y, z):
        p = 2 * np.pi
        return util.prim2cons(1 + 0.2 * np.sin(p * x + 1), 0.4 * np.sin(p * y / 0.7) + 0.1 * np.cos(p * x), 0.2 * np.sin(p * x),
                              w * np.cos(p * x), 1 + 0.1 * np.cos(p * (x + y)), cfg.gamma)
    return util.fill_state(cfg, f)


@pytest.mark.parametrize("w", [0.0, 0.2])
@pytest.mark.parametrize("stages", [1, 3])
@pytest.mark.parametrize("periodic", [(0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("nx,ny", [(2, 2), (59, 3), (60, 20), (61, 33), (62, 5), (120, 64), (122, 31)])
def test_against_oracle(nx, ny, periodic, stages, w):
    cfg = config(nx, ny, periodic, stages)
    U = flow(cfg, w)
    o, s = pyoracle.Oracle(cfg), capi.Solver(cfg)
    o.set_state(U)
    s.set_state(U)
    a, b = s.step(12), o.step(12)
    got, ref = capi.interior(cfg, s.get_state()), capi.interior(cfg, o.get_state())
    s.close()
    assert a.steps_done == b.steps_done == 12
    assert abs(a.time - b.time) <= 1e-12 * b.time
    assert util.normwise_rel(got, ref).max() <= 1e-12


@pytest.mark.parametrize("stages", [1, 3])
@pytest.mark.parametrize("periodic", [(0, 0), (1, 1)])
@pytest.mark.parametrize("nx,ny", [(2, 2), (61, 33), (120, 64)])
def test_plane_flow_in_both_forms(nx, ny, periodic, stages):
    # the momentum out of the plane is too small to reach another variable, and brings in the kernels with all
    # five; the four others' operations are the same but for what the compiler fuses, a few ulps a step
    cfg = config(nx, ny, periodic, stages)
    runs = []
    for w in (0.0, 1e-30):
        s = capi.Solver(cfg)
        s.set_state(flow(cfg, w))
        runs.append((s.step(12).time, capi.interior(cfg, s.get_state())))
        s.close()
    assert abs(runs[0][0] - runs[1][0]) <= 1e-12 * runs[0][0]
    assert util.normwise_rel(runs[1][1], runs[0][1]).max() <= 1e-12
    assert np.all(runs[0][1][..., 3] == 0.0) and np.any(runs[1][1][..., 3] != 0.0)
