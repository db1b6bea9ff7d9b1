"""Which kernels an upload chooses, on both sides of the 8192 cells up to which the host looks through the state:
momentum out of the grid's axes in a single cell, at either end, brings in all five variables (the algorithmic
bytes tell); in a ghost cell, or as a negative zero, it does not; and forward Euler, which ends in
either of its two buffers, keeps a left-out momentum at zero after a state that had one."""
import numpy as np
import pytest

from turbostructred_amd import capi
import util

pytestmark = pytest.mark.gpu

SIZES = [(8192,), (8193,), (128, 64), (241, 34)]


def config(n, stages):
    return capi.make_config(ndims=len(n), nx=n[0], ny=n[1] if len(n) > 1 else 1, cfl=0.4, riemann=capi.RIEMANN_HLLC,
                            recon=capi.RECON_LINEAR_LIM, rk_stages=stages, bcs=[dict(type=capi.BC_NATURAL)])


def plane(cfg):
    return util.fill_state(cfg, lambda x, y, z: util.prim2cons(1 + 0.2 * np.sin(6 * x), 0.3, 0.1 if cfg.ndims > 1 else 0.0,
                                                               0.0, 1.0, cfg.gamma)).reshape(capi.state_shape(cfg))


@pytest.mark.parametrize("n", SIZES)
def test_choice(n):
    cfg = config(n, 3)
    s = capi.Solver(cfg)

    def variables(U):
        s.set_state(U)
        return s.algorithmic_bytes_per_cell(capi.KIND_STAGE1) / 16

    base = plane(cfg)
    inner = (0, 0) if cfg.ndims == 1 else (0, 1)
    last = (0, 0, -2) if cfg.ndims == 1 else (0, -2, -2)
    outside = [2, 3] if cfg.ndims == 1 else [3]
    assert variables(base) == cfg.ndims + 2
    for cell in ((*inner, 1), last):
        for v in outside:
            for value in (1e-300, np.nan):
                U = base.copy()
                U[(*cell, v)] = value
                assert variables(U) == 5
    U = base.copy()
    U[..., outside] = -0.0
    assert variables(U) == cfg.ndims + 2
    U[0, 0, 0, outside] = 1.0
    U[0, -1, -1, outside] = np.nan
    assert variables(U) == cfg.ndims + 2
    s.close()


@pytest.mark.parametrize("n", SIZES)
def test_forward_euler_buffers(n):
    cfg = config(n, 1)
    U = plane(cfg)
    W = U.copy()
    W[..., 3] = 0.1
    s = capi.Solver(cfg)
    for S, steps in ((U, 3), (U, 2), (W, 3), (U, 3), (W, 2), (U, 3), (U, 3)):
        s.set_state(S)
        s.set_time(0.0, 0)
        s.step(steps)
        got = capi.interior(cfg, s.get_state())
        fresh = capi.Solver(cfg)
        fresh.set_state(S)
        fresh.step(steps)
        assert np.array_equal(got, capi.interior(cfg, fresh.get_state()))
        assert np.all((got[..., 3] == 0.0) == (S is U))
        fresh.close()
    s.close()
