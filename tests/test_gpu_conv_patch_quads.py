"""k_conv3x3_patch with two channel quads of a wavefront in LDS: sums of small whole numbers, which every order of adding gives
exactly, and the activation and pooling on them."""
from ctypes import byref

import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.test_gpu_conv_lanes import _forward

pytestmark = pytest.mark.gpu

PATCH = 2   # gh_conv_route

# B, C, H, W, F, padding: an even and an odd number of quads, the fewest, one short of it (the loop of one quad); 11 and 9
# tiles of pixels, 16 and 32 filters to a workgroup and fewer, several patches with ones that end outside the image, patches of
# 240 cells, one more column than they have, no padding
CASES = [(8, 128, 13, 13, 1024, 1), (8, 160, 13, 13, 1000, 1), (3, 96, 13, 13, 64, 1), (4, 224, 12, 12, 1024, 1), (1, 160, 12, 12, 40, 1), (2, 128, 26, 26, 250, 1),
         (5, 128, 22, 22, 256, 1), (4, 128, 8, 22, 96, 1), (4, 160, 8, 23, 96, 1), (4, 128, 15, 15, 70, 0), (2, 256, 11, 11, 17, 1), (3, 192, 24, 20, 48, 1)]


@pytest.mark.parametrize("B,C,H,W,F,pad", CASES)
def test_whole_numbers(ctx, monkeypatch, B, C, H, W, F, pad):
    for other in ("LANES", "ROWS", "SMALL"):
        monkeypatch.setenv("GORGONIA_HIP_CONV_NO_" + other, "1")
    rng = np.random.default_rng(C + H + F)
    w, x = rng.integers(-3, 4, (F, C, 3, 3)).astype(np.float32), rng.integers(-4, 5, (B, C, H, W)).astype(np.float32)
    y = _forward(x, w, pad)[:, :, :, 1 - pad:W - 1 + pad]
    oh, ow = y.shape[2:]
    px, pw = ctx.upload(x), ctx.upload(w)
    for kw in ({}, dict(act="relu", pool2=True)):
        want = y if not kw else np.maximum(y, 0)[:, :, :oh // 2 * 2, :ow // 2 * 2].reshape(B, F, oh // 2, 2, ow // 2, 2).max((3, 5))
        out = ctx.upload(np.full(want.size + 64, np.nan, np.float32))
        cmd = D.cmd_conv2d(px, pw, out, B, C, H, W, F, 3, 3, (pad, pad), **kw)
        if not kw or ctx.lib.gh_conv2d_can_pool(byref(cmd)):
            assert ctx.lib.gh_conv2d_route(byref(cmd)) == PATCH
            ctx.run(cmd)
            got = ctx.d2h(out, (want.size + 64,))
            assert np.array_equal(got[:want.size].reshape(want.shape), want) and np.isnan(got[want.size:]).all(), kw
        ctx.free(out)
    ctx.free(px)
    ctx.free(pw)
