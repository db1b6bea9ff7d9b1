"""Algorithmic bytes of the kernels in use: the variables they carry, which a state without momentum out of the
grid's axes reduces and any other state brings back; and where the stages form the viscous fluxes, the bytes
of those stages beside their time."""
import numpy as np
import pytest

from turbostructred_amd import capi
import util

pytestmark = pytest.mark.gpu

KINDS = [capi.KIND_DT, capi.KIND_STAGE1, capi.KIND_STAGE2, capi.KIND_STAGE3, capi.KIND_ALL, capi.KIND_VISCOUS]
# arrays of doubles (d) and of the working type (s) that the kinds read and write: FP64, then FP32 residual
EULER = ([(1, 0), (2, 0), (0, 0), (0, 0)],) * 2
RK3 = [(0, 0), (1, 1), (1, 2), (2, 1)], [(0, 0), (1, 1), (1, 3), (2, 2)]
RK3_SEPARATE = [(1, 0), (1, 1), (1, 2), (2, 1)]


def arrays(table, planes, real):
    b = [planes * (8 * d + real * s) for d, s in table]
    return b + [sum(b)]


def counted(nd, stages, precision, w, **kw):
    n = dict(zip(("nx", "ny", "nz"), (24, 18, 12)[:nd]))
    cfg = capi.make_config(ndims=nd, cfl=0.4, riemann=capi.RIEMANN_ROE, recon=capi.RECON_LINEAR_LIM, rk_stages=stages,
                           precision=precision, bcs=[dict(type=capi.BC_NATURAL)], **n, **kw)
    s = capi.Solver(cfg)
    out = []
    for wk in w:
        s.set_state(util.fill_state(cfg, lambda x, y, z: util.prim2cons(1 + 0.1 * np.sin(6 * x), 0.3, 0.0, wk, 1.0, cfg.gamma)))
        out.append([s.algorithmic_bytes_per_cell(k) for k in KINDS])
    s.close()
    return out


@pytest.mark.parametrize("precision", [capi.FP64, capi.FP32_RESIDUAL])
@pytest.mark.parametrize("stages", [1, 3])
@pytest.mark.parametrize("nd", [1, 2, 3])
def test_variables_in_use(nd, stages, precision):
    fp32 = precision == capi.FP32_RESIDUAL
    table = (EULER if stages == 1 else RK3)[fp32]
    for got, planes in zip(counted(nd, stages, precision, (0.0, 0.2, 0.0)), (nd + 2, 5, nd + 2)):
        assert got == arrays(table, planes, 4 if fp32 else 8) + [0.0]


@pytest.mark.parametrize("stages", [1, 3])
def test_viscous_stages(stages):
    table = EULER[0] if stages == 1 else RK3_SEPARATE
    for got, planes in zip(counted(2, stages, capi.FP64, (0.0, 0.2), viscous=True, viscosity=0.01), (4, 5)):
        b = arrays(table, planes, 8)
        assert got == b + [pytest.approx(sum(b[1:4]) / stages)]
