"""k_conv3x3_lanes by workgroups that have several tiles each: on a context that plans for one to three compute units, sums of
small whole numbers, which every order of adding gives exactly, and the activation and pooling on them."""
from ctypes import byref

import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.test_gpu_conv_lanes import _forward

pytestmark = pytest.mark.gpu

# B, C, H, W, F and the numbers of compute units that it is planned for: tiles of whole filters and rows and short of one, one
# quad to a wavefront, several and none; and the forms that run so (100 x wavefronts + 10 x filter tiles + whether they split the
# channels) of the convolution, of it pooled and of the image gradient
CASES = [("f32", (1, 64, 26, 26, 128, range(4, 60, 3)), {811}, {811}, {811, 821}), ("f32", (2, 24, 22, 24, 40, range(2, 30, 2)), (), (), {811}),
         ("f32", (3, 16, 40, 41, 32, range(2, 40, 3)), (), (), {811}), ("f32", (2, 8, 60, 60, 16, range(4, 40, 4)), (), (), {811}),
         ("f32", (2, 128, 26, 26, 256, range(20, 150, 8)), {821}, {821}, {811, 821}), ("f32", (2, 96, 30, 30, 96, range(5, 120, 8)), {421}, {421}, {811, 821}),
         ("f32", (6, 256, 10, 10, 256, range(20, 256, 16)), {421, 811, 821}, {421, 811, 821}, {811, 821}), ("f32", (10, 32, 104, 104, 64, [256]), {410}, {410}, ()),
         ("f64", (1, 64, 26, 26, 128, range(4, 60, 3)), {411, 420, 421}, (), {411, 421}), ("f64", (2, 24, 22, 24, 40, range(2, 30, 2)), {411}, (), {411, 421}),
         ("f64", (3, 16, 40, 41, 32, range(2, 40, 3)), {411, 420}, (), {411}), ("f64", (2, 8, 60, 60, 16, range(4, 40, 4)), {411}, (), ()),
         ("f64", (9, 32, 8, 8, 64, range(1, 20)), {411, 421}, (), {411, 421})]


@pytest.mark.parametrize("dt,case,plain,pooled,gradient", CASES)
def test_whole_numbers(monkeypatch, dt, case, plain, pooled, gradient):
    B, C, H, W, F, units = case
    np_dt, code = (np.float32, _ffi.F32) if dt == "f32" else (np.float64, _ffi.F64)
    rng = np.random.default_rng(C + H + F)
    w = rng.integers(-3, 4, (F, C, 3, 3)).astype(np_dt)
    x, dy = rng.integers(-4, 5, (B, C, H, W)).astype(np_dt), rng.integers(-4, 5, (B, F, H, W)).astype(np_dt)
    y, dx = _forward(x, w, 1), _forward(dy, w[:, :, ::-1, ::-1].transpose(1, 0, 2, 3), 1)
    forms = set()
    for n in units:
        monkeypatch.setenv("GORGONIA_HIP_COMPUTE_UNITS", str(n))
        with D.Context(0, 0) as ctx:
            px, pw, pdy = ctx.upload(x), ctx.upload(w), ctx.upload(dy)
            todo = [(D.cmd_conv2d, {}, px, y), (D.cmd_conv2d_bwd_data, {}, pdy, dx)]
            if dt == "f32" and H % 2 == 0 and W % 2 == 0:
                todo.append((D.cmd_conv2d, dict(act="relu", pool2=True), px, np.maximum(y, 0).reshape(B, F, H // 2, 2, W // 2, 2).max((3, 5))))
            for make, kw, src, want in todo:
                out = ctx.upload(np.full(want.shape, np.nan, np_dt))
                cmd = make(src, pw, out, B, C, H, W, F, 3, 3, (1, 1), dtype=code, **kw)
                if not kw.get("pool2") or ctx.lib.gh_conv2d_can_pool(byref(cmd)):
                    before = ctx.joint_launches(_ffi.JOINT_CONV_ROUNDS)[0]
                    ctx.run(cmd)
                    after, form = ctx.joint_launches(_ffi.JOINT_CONV_ROUNDS)
                    assert np.array_equal(ctx.d2h(out, want.shape, np_dt), want), (n, make.__name__, kw)
                    if after > before:
                        forms.add((make.__name__[4:], bool(kw), form))
                ctx.free(out)
            for p in (px, pw, pdy):
                ctx.free(p)
    assert forms == {("conv2d", p, f) for p, fs in ((False, plain), (True, pooled)) for f in fs} | {("conv2d_bwd_data", False, f) for f in gradient}
