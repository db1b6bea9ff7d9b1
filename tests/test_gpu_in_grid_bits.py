"""The kernels that leave out the momenta that are zero by construction do the same operations as those that carry
them: ts_step, which chooses by the state, and ts_step_noalloc, which does not look at it, end bit for bit
alike, in each flux, reconstruction, number of stages and precision."""
import numpy as np
import pytest

import test_gpu_in_grid as forms
from turbostructred_amd import capi
import util
from test_zz_no_alloc import by_noalloc, hip_runtime, soa_interior

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("recon,lim", forms.RECONS)
@pytest.mark.parametrize("flux", [capi.RIEMANN_ROE, capi.RIEMANN_HLLC, capi.RIEMANN_GODUNOV])
@pytest.mark.parametrize("stages,precision", [(1, capi.FP64), (3, capi.FP64), (3, capi.FP32_RESIDUAL)])
@pytest.mark.parametrize("n", [(301,), (4000,), (200, 136)])
def test_same_bits(n, stages, precision, flux, recon, lim):
    nd = len(n)
    cfg = capi.make_config(ndims=nd, nx=n[0], ny=n[1] if nd > 1 else 1, cfl=0.4, riemann=flux, recon=recon, limiter=lim,
                           rk_stages=stages, precision=precision, eps=0.05 if flux == capi.RIEMANN_ROE else 0.0,
                           bcs=[dict(type=capi.BC_NATURAL), dict(type=capi.BC_WALL), dict(type=capi.BC_SYMMETRY)],
                           side_marker=(0, 1, 2, 1, 0, 0))
    states = [util.fill_state(cfg, forms.wavy(cfg.gamma, nd)), util.sod(cfg)]
    if nd == 2 and flux != capi.RIEMANN_ROE:  # (Roe's flux loses the near-vacuum quadrant)
        states.append(util.quadrants(cfg))
    for U in states:
        s = capi.Solver(cfg)
        s.set_state(U)
        ia = s.step(25)
        a = soa_interior(cfg, s.get_state()).reshape(5, -1)
        s.close()
        b, ib = by_noalloc(*hip_runtime(), cfg, U, 25)
        assert ia.steps_done == ib.steps_done == 25
        assert ia.time == ib.time and ia.dt == ib.dt
        assert np.array_equal(a, b.reshape(5, -1))
