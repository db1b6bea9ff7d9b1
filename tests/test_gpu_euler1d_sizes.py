"""1-D forward Euler in one workgroup at the sizes where it can go wrong: the fewest cells, a face
count at and beside a whole wavefront, the first size with two cells to a thread, and the last one
that stays in LDS and the first that does not, with and without transverse momentum, open and
periodic, first order and limited; the dt of every step and the state against the oracle."""
import numpy as np
import pytest

from turbostructred_amd import capi
from oracle import pyoracle
import util

pytestmark = pytest.mark.gpu

LDS = 20000  # doubles of the workgroup's arrays: (2 N + 3, + N with a reconstruction) per face


def sizes(n_var, recon):
    most = LDS // (2 * n_var + 3 + (0 if recon == capi.RECON_PWC else n_var)) - 1
    return [2, 3, 62, 63, 64, 1023, 1024, most, most + 1]


CASES = [(n_var, recon, nx) for n_var in (3, 5) for recon in (capi.RECON_PWC, capi.RECON_LINEAR_LIM)
         for nx in sizes(n_var, recon)]


@pytest.mark.parametrize("periodic", [0, 1])
@pytest.mark.parametrize("n_var,recon,nx", CASES)
def test_sizes(n_var, recon, nx, periodic):
    cfg = capi.make_config(ndims=1, nx=nx, cfl=0.4, riemann=capi.RIEMANN_ROE, eps=0.05, recon=recon, periodic=(periodic, 0, 0),
                           bcs=[dict(type=capi.BC_NATURAL), dict(type=capi.BC_WALL)], side_marker=(0, 1, 0, 0, 0, 0))

    def wave(x, y, z):
        t = 0.2 if n_var == 5 else 0.0
        return util.prim2cons(1 + 0.3 * np.sin(2 * np.pi * x), 0.2 * np.cos(2 * np.pi * x), t * np.sin(4 * np.pi * x),
                              -t * np.cos(2 * np.pi * x), 1 + 0.1 * np.cos(2 * np.pi * x), cfg.gamma)

    U = util.fill_state(cfg, wave)
    o = pyoracle.Oracle(cfg)
    o.set_state(U)
    s = capi.Solver(cfg)
    s.set_state(U)
    s.enable_dt_log(16)
    dts = []
    for _ in range(9):
        dts.append(o.step(1).dt)
    s.step(4)  # an even, then an odd number of steps: the state changes buffers in between
    info = s.step(5)
    assert info.steps_done == 5 and info.iteration == 9
    a, b = capi.interior(cfg, s.get_state()), capi.interior(cfg, o.get_state())
    log = s.dt_log(16)
    s.close()
    np.testing.assert_allclose(log, dts, rtol=1e-12)
    assert util.normwise_rel(a, b).max() <= 1e-12
