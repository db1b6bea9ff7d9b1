"""The Euler equations are homogeneous of degree one in the conserved variables: a state in other units of mass, a
power of two times as large, gives the same run times that power, bit for bit, as long as no operation leaves
the range of its type.  Densities, momenta and energies of 1e-21 to 1e21 fit a float, their squares do
not."""
import numpy as np
import pytest

from turbostructred_amd import capi
import util

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("riemann", [capi.RIEMANN_ROE, capi.RIEMANN_HLLC, capi.RIEMANN_GODUNOV])
@pytest.mark.parametrize("stages", [1, 3])
@pytest.mark.parametrize("n", [(100,), (70, 20), (20, 9, 7)])
@pytest.mark.parametrize("power", [-70, 70])
def test_units_of_mass(power, n, stages, riemann):
    nd = len(n)
    shape = dict(zip(("nx", "ny", "nz"), n))
    cfg = capi.make_config(ndims=nd, cfl=0.4, riemann=riemann, recon=capi.RECON_PWC, rk_stages=stages,
                           precision=capi.FP32_RESIDUAL, bcs=[dict(type=capi.BC_NATURAL)], **shape)
    vel = lambda q: (3.0, 0.5 + q if nd > 1 else 0.0, -0.3 if nd > 2 else 0.0)
    U = util.fill_state(cfg, lambda x, y, z: util.prim2cons(1 + 0.3 * np.sin(6 * x), *vel(0.1 * np.cos(6 * x)),
                                                            1 + 0.2 * np.cos(6 * x), cfg.gamma))
    runs = []
    for scale in (1.0, 2.0 ** power):
        s = capi.Solver(cfg)
        s.set_state(U * scale)
        info = s.step(20)
        runs.append((info.steps_done, info.time, capi.interior(cfg, s.get_state()) / scale))
        s.close()
    assert runs[0][:2] == runs[1][:2]
    assert np.array_equal(runs[0][2], runs[1][2])
