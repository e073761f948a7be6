"""A convolution's two gradients with the gradient of the pooling (and its Rectify) in front of the convolution in one launch
(k_conv_gradients.hip): the bits of the commands submitted apart, in every tensor they write and around it."""
import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.util import assert_bits_equal

pytestmark = pytest.mark.gpu

EDGE = 64
# (B, C, H, W, F): the form of the launch; every kernel that has the three, groups that overlap at a row's end, rows no group
# divides, images and filters past a tile; None: kernels that do not have them
F32 = {(128, 32, 14, 14, 64): 121, (128, 64, 7, 7, 128): 221, (3, 16, 7, 5, 40): 211, (1, 16, 16, 16, 16): 111, (37, 48, 9, 13, 72): 111, (39, 128, 8, 6, 84): 221,
       (8, 64, 26, 26, 128): None}
F64 = {(50, 32, 14, 14, 64): 411, (50, 64, 7, 7, 128): 511, (11, 32, 15, 8, 12): 511, (3, 40, 45, 11, 8): 411, (2, 16, 9, 11, 12): None}
CASES = [(np.float32,) + c for c in F32] + [(np.float64,) + c for c in F64]


def _run(ctx, dt, B, C, H, W, F, layout, want, image_first=False, big=2):
    """layout(pointers by name) -> overrides of them; all three or four commands together and apart."""
    rng = np.random.default_rng(B * C + H * W + F)
    code = _ffi.F64 if dt == np.float64 else _ffi.F32
    shape = (B, C, big * H, big * W)
    z = (np.round(rng.standard_normal(shape) * 2) / 2).astype(dt)   # ties inside windows
    z.reshape(-1)[:9] = [0.0, -0.0, np.inf, -np.inf, np.nan, np.nan, -1.0, -2.0, 1e-45]
    with np.errstate(invalid="ignore"):
        a = z * (z >= 0)
    held = {"x": rng.standard_normal((B, C, H, W)), "dy": rng.standard_normal((B, F, H, W)), "w": rng.standard_normal((F, C, 3, 3)), "z": z, "a": a}
    sizes = {"dw": F * C * 9, "dx": B * C * H * W, "da": z.size, "dz": z.size}
    got = []
    for together in (True, False):
        at = {k: ctx.upload(np.concatenate([np.full(EDGE, np.nan, dt), v.astype(dt).ravel(), np.full(EDGE, np.nan, dt)])) for k, v in held.items()}
        at.update({k: ctx.upload(np.full(n + 2 * EDGE, np.nan, dt)) for k, n in sizes.items()})
        p = {k: v + EDGE * np.dtype(dt).itemsize for k, v in at.items()}
        p.update(layout(p))
        cmds = [D.cmd_conv2d_bwd_filter(p["x"], p["dy"], p["dw"], B, C, H, W, F, 3, 3, (1, 1), dtype=code),
                D.cmd_conv2d_bwd_data(p["dy"], p["w"], p["dx"], B, C, H, W, F, 3, 3, (1, 1), dtype=code)]
        if image_first:
            cmds.reverse()
        pool = D.cmd_maxpool2d_bwd(p["z"] if dt == np.float32 else p["a"], p["dx"], p["dz"] if dt == np.float32 else p["da"], B, C, shape[2], shape[3], 2, 2, (0, 0), (2, 2),
                                   dtype=code)
        cmds.append(pool)
        if dt == np.float32:
            pool.flags |= _ffi.FLAG_ACT_RELU
        else:
            cmds.append(D.cmd_relu_bwd(p["z"], p["da"], p["dz"], z.size, dtype=code))
        if together:
            before = ctx.joint_launches(_ffi.JOINT_UNPOOLED)[0]
            ctx.run(cmds)
            after, form = ctx.joint_launches(_ffi.JOINT_UNPOOLED)
            assert after - before == (want is not None) and want in (None, form)
        else:
            for c in cmds:
                ctx.run([c])
        got.append({k: ctx.d2h(v, ((held[k].size if k in held else sizes[k]) + 2 * EDGE,), dt) for k, v in at.items()})
        for v in at.values():
            ctx.free(v)
    for k in got[0]:
        assert_bits_equal(got[0][k], got[1][k])


@pytest.mark.parametrize("image_first", [False, True])
@pytest.mark.parametrize("dt,B,C,H,W,F", CASES)
def test_with_the_pooling_in_front(ctx, dt, B, C, H, W, F, image_first):
    _run(ctx, dt, B, C, H, W, F, lambda p: {}, (F32 if dt == np.float32 else F64)[B, C, H, W, F], image_first)


@pytest.mark.parametrize("B,C,H,W,F", [(50, 64, 7, 7, 128), (11, 32, 15, 8, 12)])
def test_rectify_gradient_in_place(ctx, B, C, H, W, F):
    _run(ctx, np.float64, B, C, H, W, F, lambda p: {"da": p["dz"]}, F64[B, C, H, W, F])


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_what_overlaps_runs_apart(ctx, dt):
    """The pooling's gradient over its own input, or over what the convolution's gradients still read: as submitted apart."""
    shape = (50, 32, 14, 14, 64)
    _run(ctx, dt, *shape, lambda p: {"dz": p["z"]}, None)
    _run(ctx, dt, *shape, lambda p: {"dy": p["dz"] + EDGE * np.dtype(dt).itemsize}, None)
    _run(ctx, dt, *shape, lambda p: {"x": p["dz"]}, None)
