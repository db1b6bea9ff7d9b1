"""The checks of test_gpu_step_dt on both sides of the largest grid whose stage 2 forms the step's dt itself: 1216
workgroups of four strips by 60 columns store a minimum each, and one column more takes the separate launch.
Snapshot and end-time stops inside a call, steps one by one, and a step that fails."""
import pytest

import test_gpu_step_dt as small
from turbostructred_amd import capi

pytestmark = pytest.mark.gpu

SHAPES = [dict(ndims=1, nx=1216 * 4 * 60), dict(ndims=1, nx=1216 * 4 * 60 + 1)]


@pytest.mark.parametrize("precision", [capi.FP64, capi.FP32_RESIDUAL])
@pytest.mark.parametrize("shape", SHAPES)
def test_stops_and_dt(shape, precision):
    small.test_stops_and_dt(shape, precision)


@pytest.mark.parametrize("shape", SHAPES)
def test_failed_step(shape):
    small.test_failed_step(shape)
