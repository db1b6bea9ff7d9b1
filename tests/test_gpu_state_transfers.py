"""States come back as they went up, to the bit: sizes beside those from which several threads share a
download (24 MiB) and an upload (64 MiB) and below which a batch gathers states (4 MiB); through a
solver, and through a batch that mixes them with solves small enough to share one copy."""
import numpy as np
import pytest

from turbostructred_amd import capi
import util

pytestmark = pytest.mark.gpu

# (nx + 2) * 40 bytes: just below and at 4 MiB, 8 MiB, just below and at 24 MiB, just below and at 64 MiB
TUBES = [7, 104855, 104856, 209714, 629143, 629144, 1677719, 1677720]


def problem(nx, ny, seed, **kw):
    cfg = capi.make_config(ndims=1 + (ny > 1), nx=nx, ny=ny, cfl=0.4, riemann=capi.RIEMANN_HLLC, recon=capi.RECON_LINEAR_LIM,
                           rk_stages=3, periodic=(1, 1, 0), **kw)
    r = np.random.default_rng(seed)
    U = util.prim2cons(r.uniform(0.5, 1.5, nx * ny), r.uniform(-1, 1, nx * ny), r.uniform(-1, 1, nx * ny), 0.0,
                       r.uniform(0.5, 1.5, nx * ny), cfg.gamma)
    state = np.zeros(capi.state_shape(cfg))
    capi.interior(cfg, state)[...] = U.reshape(1, ny, nx, 5)
    return cfg, state


@pytest.mark.parametrize("nx,ny", [(n, 1) for n in TUBES] + [(700, 701)])
def test_solver(nx, ny):
    cfg, U = problem(nx, ny, nx)
    s = capi.Solver(cfg)
    for _ in range(2):  # the second time in a buffer that is there
        s.set_state(U)
        got = s.get_state()
        assert np.array_equal(capi.interior(cfg, got), capi.interior(cfg, U))
    s.close()


def test_batch():
    sizes = [(n, 1) for n in TUBES] + [(700, 701), (300, 200)] + [(20 + i % 50, 1) for i in range(300)]
    work = [problem(nx, ny, i) for i, (nx, ny) in enumerate(sizes)]
    order = np.random.default_rng(1).permutation(len(work))
    b = capi.Batch(hbm_budget_bytes=1 << 30)
    for _ in range(2):
        tickets = {int(i): b.submit(*work[i], 0) for i in order}  # no steps: the state as it was
        while b.run(4) > 0:
            pass
        for i, (cfg, U) in enumerate(work):
            done, got, info = b.poll(tickets[i])
            assert done and info.steps_done == 0
            assert np.array_equal(capi.interior(cfg, got), capi.interior(cfg, U))
    b.close()
