"""k_conv3x3_lanes at shapes that its dispatch gives it in each precision: the geometries of tests/test_gpu_conv_lanes.py
whose small float64 (and two float32) forms go to the staged kernels, with as many images and channels as it takes."""
import ctypes

import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.test_gpu_conv_lanes import _forward, _run
from tests.util import rel_frobenius

pytestmark = pytest.mark.gpu

# B, C, H, W, F, padH
F32_CASES = [(1, 128, 7, 7, 130, 1), (16, 264, 10, 10, 96, 1)]
F64_CASES = [(8, 32, 30, 4, 16, 1), (8, 24, 21, 5, 35, 1), (1, 80, 17, 18, 33, 0), (3, 72, 9, 19, 16, 2), (4, 128, 13, 13, 100, 1),
             (4, 40, 4, 33, 48, 0), (8, 64, 7, 7, 130, 1), (4, 264, 10, 10, 48, 1)]


@pytest.mark.parametrize("dt,cfg", [("f32", c) for c in F32_CASES] + [("f64", c) for c in F64_CASES])
def test_shapes_that_run_on_it(ctx, dt, cfg):
    B, C, H, W, F, padH = cfg
    code = _ffi.F32 if dt == "f32" else _ffi.F64
    bar = 2e-6 if dt == "f32" else 1e-14   # sums of at most 9 x 264 products in the operands' own precision
    args = (0x10000, 0x20000, 0x30000, B, C, H, W, F, 3, 3, (padH, 1))
    assert ctx.lib.gh_runs_straight(ctypes.byref(D.cmd_conv2d(*args, dtype=code))) == 1
    x, w, got = _run(ctx, cfg, dt)
    assert rel_frobenius(got, _forward(x, w, padH)) <= bar
    if F % 4 == 0:
        assert ctx.lib.gh_runs_straight(ctypes.byref(D.cmd_conv2d_bwd_data(*args, dtype=code))) == 1
        dy, w, got = _run(ctx, cfg, dt, flip=True)
        assert rel_frobenius(got, _forward(dy, w[:, :, ::-1, ::-1].transpose(1, 0, 2, 3), 2 - padH)) <= bar
