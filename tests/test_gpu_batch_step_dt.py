"""Batched 1-D solves around the sizes up to which stage 2 applies the step's dt itself: a lone tube of
64 work items, of 65, of as many as the reads of all their minima allow (their squares add up to at most 48 x
2^20) and of one more, tubes that the arrival and the leaving of a long one take from one form to the other, an
end time inside a pass, and a tube that fails in either form."""
import numpy as np
import pytest

from turbostructred_amd import capi
import util

pytestmark = pytest.mark.gpu

MOST = 7094 * 60  # cells of a lone tube whose minima stage 2 still reads


def tube(n, precision, k):
    cfg = capi.make_config(ndims=1, nx=n, cfl=0.45, riemann=capi.RIEMANN_HLLC, recon=capi.RECON_LINEAR_LIM, rk_stages=3,
                           precision=precision, bcs=[dict(type=capi.BC_NATURAL)])
    U = util.fill_state(cfg, lambda x, y, z: util.prim2cons(1 + 0.3 * np.sin(6 * x + k), 0.4 * np.cos(6 * x), 0.0, 0.0,
                                                            1 + 0.2 * np.cos(12 * x), cfg.gamma))
    return cfg, U


def alone(cfg, U, steps, t_end):
    s = capi.Solver(cfg)
    s.set_state(U)
    info = s.step(steps, t_end, t_end) if t_end else s.step(steps)
    got = capi.interior(cfg, s.get_state())
    s.close()
    return got, info


def check(b, ticket, cfg, U, steps, t_end):
    done, got, info = b.poll(ticket)
    ref, rinfo = alone(cfg, U, steps, t_end)
    assert done and info.steps_done == rinfo.steps_done and info.time == rinfo.time and info.dt == rinfo.dt
    assert np.array_equal(capi.interior(cfg, got), ref)


@pytest.mark.parametrize("precision", [capi.FP64, capi.FP32_RESIDUAL])
@pytest.mark.parametrize("graphs", [True, False])
@pytest.mark.parametrize("n", [64 * 60, 64 * 60 + 1, MOST, MOST + 1])
def test_lone_tube(n, graphs, precision):
    cfg, U = tube(n, precision, 0)
    info = alone(cfg, U, 3, 0.0)[1]
    for steps, t_end in ((7, 0.0), (100, 3.4 * info.time)):
        b = capi.Batch(hbm_budget_bytes=1 << 30, use_graphs=graphs)
        t = b.submit(cfg, U, steps, t_end)
        while b.run(4):
            pass
        check(b, t, cfg, U, steps, t_end)
        b.close()


@pytest.mark.parametrize("precision", [capi.FP64, capi.FP32_RESIDUAL])
def test_from_one_form_to_the_other(precision):
    b = capi.Batch(hbm_budget_bytes=1 << 30)
    work = [(*tube(600 + 60 * k, precision, k), 60, 0.0) for k in range(3)]
    tickets = [b.submit(*w) for w in work]
    b.run(8)
    work.append((*tube(MOST + 60, precision, 5), 21, 0.0))
    tickets.append(b.submit(*work[-1]))
    while b.run(8):
        pass
    for t, w in zip(tickets, work):
        check(b, t, *w)
    b.close()


@pytest.mark.parametrize("n", [300, MOST + 1])
def test_failing_tube(n):
    good = tube(n, capi.FP64, 1)
    cfg, U = tube(n, capi.FP64, 2)
    bad = U.copy()
    # two neighbours without a density: HLLC's wave speeds are those of the better side of a face
    bad.reshape(-1, 5)[n // 2:n // 2 + 2, 0] = np.nan
    b = capi.Batch(hbm_budget_bytes=1 << 30)
    tb, tg = b.submit(cfg, bad, 10), b.submit(*good, 10)
    while b.run(4):
        pass
    with pytest.raises(capi.TSError):
        b.poll(tb)
    check(b, tg, *good, 10, 0.0)
    b.close()
