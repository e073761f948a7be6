"""k_conv3x3_lanes where a wavefront has all channels of its own tile (few channels, many pixels): the edges of its groups and
tiles in both filter widths, against float64 sums, and the activation, normalisation and pooling on its results in
registers, to the bits of the plain result."""
from ctypes import byref

import numpy as np
import pytest

from gorgonia_amd import device as D
from tests.test_gpu_conv_lanes import _forward, _run, test_epilogues_on_the_plain_result as epilogues
from tests.util import rel_frobenius

pytestmark = pytest.mark.gpu

# B, C, H, W, F, padH: whole groups; rows whose last group is moved left by one to three columns; filters short of a tile;
# no and two rows of padding; two to eight quads; a last tile of pixels that ends inside a workgroup
CASES = [(8, 16, 104, 104, 32, 1), (8, 8, 104, 104, 16, 1), (8, 16, 101, 102, 32, 1), (8, 8, 99, 101, 24, 0), (7, 12, 90, 99, 40, 2), (3, 32, 150, 150, 32, 1),
         (16, 8, 51, 51, 24, 1), (8, 16, 60, 60, 128, 1)]


def _straight(ctx, cmd):
    return ctx.lib.gh_runs_straight(byref(cmd)) == 1


@pytest.mark.parametrize("cfg", CASES)
def test_forward_and_gradient(ctx, cfg):
    B, C, H, W, F, padH = cfg
    args = (0x10000, 0x20000, 0x30000, B, C, H, W, F, 3, 3, (padH, 1))
    ran = 0
    if _straight(ctx, D.cmd_conv2d(*args)):
        x, w, got = _run(ctx, cfg, "f32")
        assert rel_frobenius(got, _forward(x, w, padH)) <= 2e-6   # sums of at most 9 x 32 products, 9 x 128 in the gradients
        ran += 1
    if _straight(ctx, D.cmd_conv2d_bwd_data(*args)):
        dy, w, got = _run(ctx, cfg, "f32", flip=True)
        assert rel_frobenius(got, _forward(dy, w[:, :, ::-1, ::-1].transpose(1, 0, 2, 3), 2 - padH)) <= 2e-6
        ran += 1
    assert ran


@pytest.mark.parametrize("cfg", [c for c in CASES if c[0] * c[2] * c[3] * c[4] < 2e7])
def test_epilogues(ctx, cfg):
    epilogues(ctx, cfg)


# (sums that run over all channels, where the kernel of the convolution over dy splits them: 3.6, 1.3 and 1.2 times its error)
@pytest.mark.parametrize("cfg", [(13, 96, 45, 45, 48), (234, 8, 15, 15, 32), (181, 64, 13, 15, 32), (8, 16, 104, 104, 32), (16, 8, 51, 51, 24)])
def test_gradient_is_as_close_as_the_convolution_over_dy(ctx, cfg):
    B, C, H, W, F = cfg
    rng = np.random.default_rng(B)
    dy, w = rng.random((B, F, H, W), np.float32), rng.random((F, C, 3, 3), np.float32)
    mirrored = np.ascontiguousarray(w[:, :, ::-1, ::-1].transpose(1, 0, 2, 3))
    p = [ctx.upload(dy), ctx.upload(w), ctx.upload(mirrored), ctx.malloc(4 * B * C * H * W)]
    ctx.run(D.cmd_conv2d_bwd_data(p[0], p[1], p[3], B, C, H, W, F, 3, 3, pad=(1, 1)))
    got = ctx.d2h(p[3], (B, C, H, W))
    ctx.run(D.cmd_conv2d(p[0], p[2], p[3], B, F, H, W, C, 3, 3, pad=(1, 1)))
    over = ctx.d2h(p[3], (B, C, H, W))
    want = _forward(dy[:4], mirrored, 1)
    # (two orders of as many roundings differ by a few per cent)
    assert rel_frobenius(got[:4], want) <= 1.05 * rel_frobenius(over[:4], want)
    for q in p:
        ctx.free(q)
