"""A convolution's filter gradient and image gradient in one launch (k_conv_gradients.hip): the bits of the two commands
submitted apart, in both orders, and of what lies around their results."""
import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.util import assert_bits_equal

pytestmark = pytest.mark.gpu

# (B, C, H, W, F) and the kernel that runs both (gh_joint_launches), None where each has a launch: every kernel; images the small-image
# kernel holds and larger ones, rows that no chunk or group divides, filter counts past a tile, odd numbers of workgroups, one image;
# enough images that both gradients take several rounds
F32 = {
    (128, 32, 14, 14, 64): 121, (128, 64, 7, 7, 128): 221, (3, 16, 7, 5, 40): 211, (1, 16, 16, 16, 16): 111, (37, 48, 9, 13, 72): 111,
    (2, 16, 104, 104, 32): 311, (8, 64, 26, 26, 128): 321, (1, 32, 52, 52, 64): None, (3, 20, 33, 29, 36): None, (1, 12, 17, 23, 20): None,
    (5, 24, 40, 19, 68): 311, (21, 64, 14, 14, 28): 121, (39, 128, 8, 6, 84): 221, (54, 20, 12, 66, 32): 310, (14, 148, 65, 39, 20): 320,
    (20, 100, 9, 15, 20): 321}
F64 = {
    (50, 32, 14, 14, 64): 411, (50, 64, 7, 7, 128): 511, (2, 16, 9, 11, 12): None, (3, 24, 17, 8, 36): None, (1, 64, 26, 26, 128): 411,
    (9, 12, 20, 33, 20): None, (3, 40, 45, 11, 8): 411, (11, 32, 15, 8, 12): 511}
CASES = [(np.float32,) + c for c in F32] + [(np.float64,) + c for c in F64]


def test_every_kernel_is_among_the_cases():
    assert {*F32.values(), *F64.values()} == {None, 111, 121, 211, 221, 310, 320, 311, 321, 411, 511}


@pytest.mark.parametrize("image_first", [False, True])
@pytest.mark.parametrize("dt,B,C,H,W,F", CASES)
def test_both_gradients(ctx, dt, B, C, H, W, F, image_first):
    rng = np.random.default_rng(B * C + H * W + F)
    x = rng.standard_normal((B, C, H, W)).astype(dt)
    dy = rng.standard_normal((B, F, H, W)).astype(dt)
    w = rng.standard_normal((F, C, 3, 3)).astype(dt)
    dtype = _ffi.F64 if dt == np.float64 else _ffi.F32
    got = []
    for together in (True, False):
        at = [ctx.upload(a) for a in (x, dy, w)]
        edge = 64
        dw, dx = (ctx.upload(np.full(n + 2 * edge, np.nan, dt)) for n in (w.size, x.size))
        off = edge * x.itemsize
        cmds = [D.cmd_conv2d_bwd_filter(at[0], at[1], dw + off, B, C, H, W, F, 3, 3, (1, 1), dtype=dtype),
                D.cmd_conv2d_bwd_data(at[1], at[2], dx + off, B, C, H, W, F, 3, 3, (1, 1), dtype=dtype)]
        if image_first:
            cmds.reverse()
        if together:
            before = ctx.joint_launches(_ffi.JOINT_CONV_GRADIENTS)[0]
            ctx.run(cmds)
            after, form = ctx.joint_launches(_ffi.JOINT_CONV_GRADIENTS)
            want = (F32 if dt == np.float32 else F64)[B, C, H, W, F]
            assert after - before == (want is not None) and want in (None, form)
        else:
            for c in cmds:
                ctx.run([c])
        got.append([ctx.d2h(dw, (w.size + 2 * edge,), dt), ctx.d2h(dx, (x.size + 2 * edge,), dt)])
        for p in at + [dw, dx]:
            ctx.free(p)
    for a, b in zip(*got):
        assert_bits_equal(a, b)
        assert np.isnan(a[:edge]).all() and np.isnan(a[-edge:]).all() and not np.isnan(a[edge:-edge]).any()


def test_result_that_the_other_reads(ctx):
    """An image gradient that overwrites the images the filter gradient read, and one over the new filter: as submitted apart."""
    B, C, F, H = 16, 32, 32, 14
    rng = np.random.default_rng(5)
    x, dy = (rng.standard_normal((B, 32, H, H)).astype(np.float32) for _ in range(2))
    w = rng.standard_normal((F, C, 3, 3)).astype(np.float32)
    for which in (0, 2):
        got = []
        for together in (True, False):
            at = [ctx.upload(a) for a in (x, dy, w)]
            spare = ctx.upload(np.zeros_like(w if which == 0 else x))
            dw, dx = (spare, at[0]) if which == 0 else (at[2], spare)
            cmds = [D.cmd_conv2d_bwd_filter(at[0], at[1], dw, B, C, H, H, F, 3, 3, (1, 1)),
                    D.cmd_conv2d_bwd_data(at[1], at[2], dx, B, C, H, H, F, 3, 3, (1, 1))]
            if together:
                ctx.run(cmds)
            else:
                for c in cmds:
                    ctx.run([c])
            got.append([ctx.d2h(dw, w.shape, np.float32), ctx.d2h(dx, x.shape, np.float32)])
            for p in at + [spare]:
                ctx.free(p)
        for a, b in zip(*got):
            assert_bits_equal(a, b)


def test_tuning_switch(ctx, monkeypatch):
    """GORGONIA_HIP_CONV_APART: a launch each."""
    B, C, H, F = 2, 16, 9, 20
    at = [ctx.upload(np.ones(n, np.float32)) for n in (B * C * H * H, B * F * H * H, F * C * 9, F * C * 9, B * C * H * H)]
    cmds = [D.cmd_conv2d_bwd_filter(at[0], at[1], at[3], B, C, H, H, F, 3, 3, (1, 1)), D.cmd_conv2d_bwd_data(at[1], at[2], at[4], B, C, H, H, F, 3, 3, (1, 1))]
    monkeypatch.setenv("GORGONIA_HIP_CONV_APART", "1")
    before = ctx.joint_launches(_ffi.JOINT_CONV_GRADIENTS)
    ctx.run(cmds)
    assert ctx.joint_launches(_ffi.JOINT_CONV_GRADIENTS) == before
    monkeypatch.delenv("GORGONIA_HIP_CONV_APART")
    ctx.run(cmds)
    assert ctx.joint_launches(_ffi.JOINT_CONV_GRADIENTS) == (before[0] + 1, 111)
    for p in at:
        ctx.free(p)
