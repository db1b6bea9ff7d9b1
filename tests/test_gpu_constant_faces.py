"""The exact solver's short way for faces with the same state on both sides is taken by a wavefront as a whole,
or lane by lane where other faces share the wavefront: a face's flux and wave speed are the same bits
either way.  A flow that is uniform but for one corner keeps the bits of every cell the corner does not
reach in the step, also between a row of faces that is wholly uniform and one that is not; and a denser
end of a tube, whose waves are slower, leaves the dt of the uniform tube."""
import numpy as np
import pytest

from turbostructred_amd import capi
import util

pytestmark = pytest.mark.gpu

STATES = np.random.default_rng(7).uniform((0.1, -2.0, -2.0, -2.0, 0.1), (2.0, 2.0, 2.0, 2.0, 3.0), (40, 5))


def config(n, stages, precision, cfl=0.4):
    shape = dict(zip(("nx", "ny", "nz"), n))
    return capi.make_config(ndims=len(n), cfl=cfl, riemann=capi.RIEMANN_GODUNOV, recon=capi.RECON_PWC, rk_stages=stages,
                            precision=precision, bcs=[dict(type=capi.BC_NATURAL)], **shape)


def uniform(cfg, state):
    vel = [state[1 + a] if a < cfg.ndims else 0.0 for a in range(3)]
    U = util.fill_state(cfg, lambda x, y, z: util.prim2cons(state[0] + 0 * x, *vel, state[4], cfg.gamma))
    return U.astype(np.float32).astype(np.float64)  # forward Euler adds to the float form of the state


@pytest.mark.parametrize("precision", [capi.FP64, capi.FP32_RESIDUAL])
@pytest.mark.parametrize("n", [(50, 20), (130, 20), (50, 8, 9)])
def test_cells_beside_uniform_rows(n, precision):
    # a step long enough that a difference in the last bit of a flux reaches the state
    cfg = config(n, 1, precision, cfl=20.0)
    far = tuple(slice(m // 2 - 1 if a < len(n) else 0, None) for a, m in reversed(list(enumerate((*n, 1, 1)[:3]))))
    changed = []
    for k, state in enumerate(STATES):
        U = uniform(cfg, state).reshape(capi.state_shape(cfg))
        corner = tuple(slice(m // 2 + 1, None) for m in reversed(n))
        U[(0,) * (3 - len(n)) + corner][..., 4] *= 1.5  # more pressure
        s = capi.Solver(cfg)
        s.set_state(U)
        assert s.step(1).steps_done == 1
        got, ref = capi.interior(cfg, s.get_state()), capi.interior(cfg, U)
        s.close()
        out = np.ones(got.shape[:3], bool)
        out[far] = False
        assert not np.array_equal(got, ref)
        if not np.array_equal(got[out], ref[out]):
            changed.append(k)
    assert changed == []


@pytest.mark.parametrize("stages", [1, 3])
@pytest.mark.parametrize("n", [(120,), (3000,)])
def test_dt_beside_a_denser_end(n, stages):
    cfg = config(n, stages, capi.FP64)
    differ = []
    for k, state in enumerate(STATES):
        state = np.abs(state)  # to the right, so that the waves at the contact are slower than u + a
        dt = []
        for dense in (False, True):
            U = uniform(cfg, state).reshape(-1, 5)
            if dense:
                U[n[0] - 20:, :2] *= 4
                U[n[0] - 20:, 4] += 1.5 * state[0] * state[1] ** 2
            s = capi.Solver(cfg)
            s.set_state(U)
            dt.append(s.step(1).dt)
            s.close()
        if dt[0] != dt[1]:
            differ.append(k)
    assert differ == []
