"""The exact solver takes a shorter way where every face of a wavefront has the same state on both
sides: uniform flows at rest, subsonic and supersonic stay bitwise as they are with the oracle's dt,
and a jump at either end of a tube, which leaves some wavefronts constant and others not, follows
the oracle.  Sizes at and beside the 60 columns of a wavefront."""
import numpy as np
import pytest

from turbostructred_amd import capi
from oracle import pyoracle
import util

pytestmark = pytest.mark.gpu
SIZES = {1: [(2,), (59,), (60,), (61,), (200,)], 2: [(61, 5), (130, 3)], 3: [(61, 4, 4)]}


def config(n, precision):
    n = tuple(n) + (1,) * (3 - len(n))
    nd = 1 + (n[1] > 1) + (n[2] > 1)
    return capi.make_config(ndims=nd, nx=n[0], ny=n[1], nz=n[2], cfl=0.4, riemann=capi.RIEMANN_GODUNOV,
                            recon=capi.RECON_LINEAR_LIM, rk_stages=3, precision=precision,
                            bcs=[dict(type=capi.BC_NATURAL)])


def start(cfg, state):
    return util.fill_state(cfg, lambda x, y, z: util.prim2cons(*(np.broadcast_to(q, x.shape) for q in state(x)), cfg.gamma))


@pytest.mark.parametrize("precision", [capi.FP64, capi.FP32_RESIDUAL])
@pytest.mark.parametrize("u", [0.0, 0.25, -3.0])
@pytest.mark.parametrize("n", SIZES[1] + SIZES[2] + SIZES[3])
def test_uniform(n, u, precision):
    cfg = config(n, precision)
    # values that a float holds exactly
    U = start(cfg, lambda x: (0.5, u, 0.0, 0.0, 1.25))
    U = U.astype(np.float32).astype(np.float64)
    o, s = pyoracle.Oracle(cfg), capi.Solver(cfg)
    o.set_state(U)
    s.set_state(U)
    a, b = s.step(4), o.step(4)
    got = capi.interior(cfg, s.get_state())
    s.close()
    assert a.steps_done == 4
    # the wave speed is one rounding of the working type per operation, about ten of them
    assert abs(a.time - b.time) <= (1e-14 if precision == capi.FP64 else 2e-6) * b.time
    # every face has the same flux, so all cells stay alike; a stage may add one rounding of a face's
    # flux times its area (fluxes up to 20 here, dt S / V below 1), and there are 12 stages
    assert np.array_equal(got, np.broadcast_to(got[:1, :1, :1], got.shape))
    eps = 1.2e-16 if precision == capi.FP64 else 6e-8
    np.testing.assert_allclose(got, capi.interior(cfg, U), rtol=0, atol=12 * 20 * eps)


@pytest.mark.parametrize("at", [0.03, 0.5, 0.97])
@pytest.mark.parametrize("n", SIZES[1][1:] + SIZES[2])
def test_jump(n, at):
    cfg = config(n, capi.FP64)
    U = start(cfg, lambda x: (np.where(x < at, 1.0, 0.125), 0.1, 0.0, 0.0, np.where(x < at, 1.0, 0.1)))
    o, s = pyoracle.Oracle(cfg), capi.Solver(cfg)
    o.set_state(U)
    s.set_state(U)
    a, b = s.step(20), o.step(20)
    got, ref = capi.interior(cfg, s.get_state()), capi.interior(cfg, o.get_state())
    s.close()
    assert abs(a.time - b.time) <= 1e-12 * b.time
    assert util.normwise_rel(got, ref).max() <= 1e-12
