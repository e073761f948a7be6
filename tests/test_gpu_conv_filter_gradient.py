"""3x3 stride-1 filter gradients at the edges of the chunks, tiles and slices of k_conv3x3_wgrad, whose operands go from
memory straight to the matrix cores, against a float64 sum over shifted images.  Each shape runs on the kernel that the
dispatch finds the quicker; the shapes that must run on the one or the other are in
tests/test_gpu_conv_filter_gradient_edges.py."""
import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.util import rel_frobenius

pytestmark = pytest.mark.gpu

# B, C, H, W, F, pad: packed columns (1 to 8 channels) and channel tiles, whole and ragged; rows of one chunk, of
# several, of one more column than a chunk; rows of at most eight columns; no padding and padding wider than the
# filter's reach; a single row; fewer chunks than wavefronts and several slices
CASES = [
    (2, 3, 101, 83, 16, 1), (1, 4, 134, 128, 20, 0), (2, 2, 90, 97, 8, 2), (2, 5, 40, 33, 9, 1), (1, 8, 37, 64, 40, 1),
    (2, 7, 31, 17, 33, 3), (1, 16, 52, 52, 32, 1), (2, 17, 20, 31, 48, 0), (1, 24, 33, 16, 16, 1), (1, 9, 20, 18, 17, 1),
    (1, 64, 40, 48, 128, 1), (4, 20, 17, 8, 50, 1), (6, 33, 30, 7, 31, 1), (3, 16, 64, 9, 64, 0), (1, 12, 1, 300, 16, 1),
    (1, 40, 300, 1, 24, 1), (1, 16, 16, 17, 8, 1), (8, 16, 104, 104, 32, 1),
]
F64_CASES = CASES[:-1] + [(20, 1, 28, 28, 32, 1), (10, 32, 14, 14, 64, 1), (10, 64, 7, 7, 128, 1)]


def _reference(x, dy, pad):
    B, C, H, W = x.shape
    F, oh, ow = dy.shape[1:]
    xp = np.zeros((B, C, H + 2 * pad, W + 2 * pad))
    xp[:, :, pad:pad + H, pad:pad + W] = x
    out = np.empty((F, C, 3, 3))
    d = dy.astype(np.float64).transpose(1, 0, 2, 3).reshape(F, -1)
    for ky in range(3):
        for kx in range(3):
            out[:, :, ky, kx] = d @ xp[:, :, ky:ky + oh, kx:kx + ow].transpose(1, 0, 2, 3).reshape(C, -1).T
    return out


@pytest.fixture(scope="module")
def ctx():
    c = D.Context(0, 0)
    yield c
    c.close()


def _run(ctx, cfg, np_dt, code):
    B, C, H, W, F, pad = cfg
    rng = np.random.default_rng(B * 1000 + C * 10 + W)
    oh, ow = H + 2 * pad - 2, W + 2 * pad - 2
    x = rng.uniform(-1, 1, (B, C, H, W)).astype(np_dt)
    dy = rng.uniform(-1, 1, (B, F, oh, ow)).astype(np_dt)
    cmd_of = lambda p, q, r: D.cmd_conv2d_bwd_filter(p, q, r, B, C, H, W, F, 3, 3, (pad, pad), dtype=code)  # noqa: E731
    px, pg, pw = ctx.upload(x), ctx.upload(dy), ctx.upload(np.full((F, C, 3, 3), np.nan, np_dt))
    ctx.run(cmd_of(px, pg, pw))
    got = ctx.d2h(pw, (F, C, 3, 3), np_dt)
    ctx.run(cmd_of(px, pg, pw))
    again = ctx.d2h(pw, (F, C, 3, 3), np_dt)
    for p in (px, pg, pw):
        ctx.free(p)
    assert np.array_equal(got, again)
    return got, _reference(x, dy, pad), ctx.lib.gh_conv2d_bwd_filter_route(cmd_of(1, 1, 1))


@pytest.mark.parametrize("cfg", CASES)
def test_float32(ctx, cfg):
    got, want, route = _run(ctx, cfg, np.float32, _ffi.F32)
    assert route == 2
    # a float32 sum over up to 86528 products in some hundred partial sums: the worst case is (chain length) 2^-24
    # of the absolute sum, random signs leave the root of it; the engine's bar for products is 1e-5
    assert rel_frobenius(got, want) <= 1e-5


@pytest.mark.parametrize("cfg", F64_CASES)
def test_float64(ctx, cfg):
    got, want, _ = _run(ctx, cfg, np.float64, _ffi.F64)
    assert rel_frobenius(got, want) <= 1e-13
