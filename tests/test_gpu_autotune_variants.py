"""The autotuner keeps the kernels of a plane flow and those with every variable apart: a tile height measured
on the former is not the height of contexts that can only run the latter, and the other way round; without a
caller's state it serves both.  The height shows in the memory of a context, which holds one double per
workgroup: the grids tuned here have two rows, so heights of at most two, in the table's size class of a grid whose
own choice is far higher."""
import numpy as np
import pytest

from turbostructred_amd import capi
import util

pytestmark = pytest.mark.gpu


def config(nx, ny, flux, out_of_plane=0.0):
    return capi.make_config(ndims=2, nx=nx, ny=ny, cfl=0.4, riemann=flux, recon=capi.RECON_LINEAR, rk_stages=3,
                            bcs=[dict(type=capi.BC_NATURAL),
                                 dict(type=capi.BC_MOVING_WALL, velocity=(0.0, 0.0, out_of_plane))])


def footprint(cfg):
    s = capi.Solver(cfg)
    out = s.footprint()
    s.close()
    return out


def state(cfg, w):
    return util.fill_state(cfg, lambda x, y, z: util.prim2cons(1 + 0 * x, 0.1, 0.0, w, 1.0, cfg.gamma))


@pytest.mark.parametrize("w", [0.0, 0.2])
def test_kept_apart(w):
    flux = capi.RIEMANN_HLLC if w else capi.RIEMANN_ROE  # a table entry for each
    small = config(1 << 21, 2, flux)
    every = config(2048, 2048, flux, out_of_plane=0.1)  # no reduced kernels
    before = footprint(every)
    chosen, cands = capi.autotune_state(small, state(small, w), steps=2)
    assert chosen <= 2 and len(cands) == 2
    assert (footprint(every) == before) == (w == 0.0)


def test_without_a_state():
    flux = capi.RIEMANN_GODUNOV
    every = config(2048, 2048, flux, out_of_plane=0.1)
    before = footprint(every)
    assert capi.autotune(config(1 << 21, 2, flux))[0] <= 2
    assert footprint(every) > before
