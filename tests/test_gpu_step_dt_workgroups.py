"""The dt of a step from one minimum per workgroup of four tiles: tile counts that fill the last workgroup
and that leave one to three of its wavefronts without a tile, 64 and 640 workgroups (one load a lane, and
one round trip) and one more, the most whose minima stage 2 reduces itself (1216) and one more, with the cell that limits dt in the first, a middle and the last tile,
for fused SSP-RK3 and for forward Euler's dt pass."""
import numpy as np
import pytest

from turbostructred_amd import capi
from oracle import pyoracle
import util

pytestmark = pytest.mark.gpu

SIZES = [(60, 1), (61, 1), (180, 1), (241, 1), (130, 7), (301, 9)] + [(4 * 60 * w + d, 1) for w in (64, 640, 1216) for d in (0, 1)]


@pytest.mark.parametrize("stages", [1, 3])
@pytest.mark.parametrize("at", [0.0, 0.4, 1.0])
@pytest.mark.parametrize("nx,ny", SIZES)
def test_dt(nx, ny, at, stages):
    cfg = capi.make_config(ndims=1 + (ny > 1), nx=nx, ny=ny, cfl=0.4, riemann=capi.RIEMANN_HLLC, recon=capi.RECON_LINEAR_LIM,
                           rk_stages=stages, bcs=[dict(type=capi.BC_NATURAL)])
    U = util.fill_state(cfg, lambda x, y, z: util.prim2cons(1 + 0 * x, 0.1, 0.0, 0.0, 1.0, cfg.gamma))
    inner = capi.interior(cfg, U)
    j, i = int(at * (ny - 1)), int(at * (nx - 1))
    inner[0, j, i, 4] *= 9.0  # three times the sound speed
    o, s = pyoracle.Oracle(cfg), capi.Solver(cfg)
    o.set_state(U)
    s.set_state(U)
    s.enable_dt_log(4)
    s.step(3)
    dts = [o.step(1).dt for _ in range(3)]
    log = s.dt_log(4)
    got, ref = capi.interior(cfg, s.get_state()), capi.interior(cfg, o.get_state())
    s.close()
    np.testing.assert_allclose(log, dts, rtol=1e-12)
    assert util.normwise_rel(got, ref).max() <= 1e-12
