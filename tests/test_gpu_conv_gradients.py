"""A convolution's filter gradient and image gradient in one launch (k_conv_gradients.hip): the bits of the two commands
submitted apart, in both orders, and of what lies around their results."""
import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.util import assert_bits_equal

pytestmark = pytest.mark.gpu

# (B, C, H, W, F): images the small-image kernel holds and larger ones, rows that no chunk or group divides, filter counts past
# a tile, odd numbers of workgroups, one image; enough images that both gradients take several rounds
F32 = [(128, 32, 14, 14, 64), (128, 64, 7, 7, 128), (3, 16, 7, 5, 40), (1, 16, 16, 16, 16), (37, 48, 9, 13, 72), (2, 16, 104, 104, 32), (8, 64, 26, 26, 128),
       (1, 32, 52, 52, 64), (3, 20, 33, 29, 36), (1, 12, 17, 23, 20), (5, 24, 40, 19, 68)]
F64 = [(50, 32, 14, 14, 64), (50, 64, 7, 7, 128), (2, 16, 9, 11, 12), (3, 24, 17, 8, 36), (1, 64, 26, 26, 128), (9, 12, 20, 33, 20)]
CASES = [(np.float32,) + c for c in F32] + [(np.float64,) + c for c in F64]


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
            ctx.run(cmds)
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
