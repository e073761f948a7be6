"""The 3x3 stride-1 filter gradient where a value must not be touched: infinities and NaN beside the columns a row
does not have, and images of a handful of values.  Against the sum over shifted, zero-padded images in float64, in
which such a value reaches the taps that read it and no other."""
import ctypes

import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.util import rel_frobenius

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = D.Context(0, 0)
    yield c
    c.close()


def _reference(x, dy, pad):
    B, C, H, W = x.shape
    F, oh, ow = dy.shape[1:]
    xp = np.zeros((B, C, H + 2 * pad[0], W + 2 * pad[1]))
    xp[:, :, pad[0]:pad[0] + H, pad[1]:pad[1] + W] = x
    out = np.empty((F, C, 3, 3))
    d = dy.astype(np.float64).transpose(1, 0, 2, 3).reshape(F, -1)
    for ky in range(3):
        for kx in range(3):
            out[:, :, ky, kx] = d @ xp[:, :, ky:ky + oh, kx:kx + ow].transpose(1, 0, 2, 3).reshape(C, -1).T
    return out


def _compare(ctx, x, dy, pad, code):
    B, C, H, W = x.shape
    F = dy.shape[1]
    px, pg, pw = ctx.upload(x), ctx.upload(dy), ctx.upload(np.full((F, C, 3, 3), np.nan, x.dtype))
    ctx.run(D.cmd_conv2d_bwd_filter(px, pg, pw, B, C, H, W, F, 3, 3, pad, dtype=code))
    got = ctx.d2h(pw, (F, C, 3, 3), x.dtype)
    for p in (px, pg, pw):
        ctx.free(p)
    with np.errstate(invalid="ignore"):
        want = _reference(x, dy, pad)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(np.isinf(got), inf) and np.array_equal(got[inf], want[inf])
    finite = np.isfinite(want)
    # the bars of the engine's products (random signs leave the root of the chain length in units of 2^-24, 2^-53)
    assert rel_frobenius(got[finite], want[finite]) <= (1e-5 if code == _ffi.F32 else 1e-13)


# B, C, H, W, F, pad: rows that end inside a chunk of 16 (8) columns, by one and by several; packed columns (up to
# eight channels) and channel tiles; no padding, and padding that puts the image's end before the row's
RAGGED = [(16, 16, 26, 26, 32, 1), (24, 32, 20, 18, 40, 0), (1, 16, 40, 52, 16, 1), (12, 16, 24, 17, 16, 2), (6, 48, 30, 19, 16, 3),
          (8, 20, 30, 18, 16, 0), (20, 16, 40, 31, 32, 1), (24, 33, 30, 7, 32, 1), (24, 48, 9, 30, 64, 1), (2, 8, 40, 37, 16, 1),
          (2, 5, 60, 35, 24, 0)]
RAGGED_F64 = RAGGED + [(8, 16, 26, 26, 32, 1), (6, 12, 30, 19, 48, 3), (12, 32, 7, 7, 16, 1), (4, 64, 14, 14, 32, 1),
                       (2, 1, 28, 28, 32, 1), (12, 16, 9, 9, 16, 0)]
# float32 channel tiles whose walk is the quicker one, and shapes that went to it before there was a choice
WALKS = RAGGED[:9] + [(16, 16, 52, 52, 32, 1), (8, 48, 20, 31, 48, 0), (24, 24, 33, 16, 16, 1), (4, 9, 60, 60, 16, 1), (8, 64, 40, 48, 64, 1),
                      (24, 32, 17, 8, 50, 1), (2, 40, 300, 1, 16, 1), (3, 12, 1, 300, 16, 1)]
STAGED = [(12, 249, 20, 20, 376, 0), (2, 16, 26, 26, 32, 1), (1, 64, 40, 48, 128, 1), (3, 26, 13, 13, 67, 1), (32, 85, 37, 6, 295, 0)]


def _route(ctx, cfg, code):
    B, C, H, W, F, pad = cfg
    cmd = D.cmd_conv2d_bwd_filter(0x1000, 0x2000, 0x3000, B, C, H, W, F, 3, 3, (pad, pad), dtype=code)
    return ctx.lib.gh_runs_straight(ctypes.byref(cmd))


@pytest.mark.parametrize("cfg", WALKS + STAGED)
def test_float32_channels(ctx, cfg):
    assert _route(ctx, cfg, _ffi.F32) == (cfg in WALKS)
    B, C, H, W, F, pad = cfg
    rng = np.random.default_rng(B * 100 + C)
    x = rng.uniform(-1, 1, (B, C, H, W)).astype(np.float32)
    dy = rng.uniform(-1, 1, (B, F, H + 2 * pad - 2, W + 2 * pad - 2)).astype(np.float32)
    _compare(ctx, x, dy, (pad, pad), _ffi.F32)


@pytest.mark.parametrize("where", ["x", "dy"])
@pytest.mark.parametrize("dt,cfg", [("f32", c) for c in RAGGED] + [("f64", c) for c in RAGGED_F64])
def test_infinities_and_nan_at_the_ends_of_rows(ctx, dt, cfg, where):
    np_dt, code = (np.float32, _ffi.F32) if dt == "f32" else (np.float64, _ffi.F64)
    assert _route(ctx, cfg, code)
    B, C, H, W, F, pad = cfg
    oh, ow = H + 2 * pad - 2, W + 2 * pad - 2
    rng = np.random.default_rng(W * 10 + pad)
    x = rng.uniform(-1, 1, (B, C, H, W)).astype(np_dt)
    dy = rng.uniform(-1, 1, (B, F, oh, ow)).astype(np_dt)
    if where == "x":   # a channel each: the last column, the one before it, the first; the other channels stay finite
        for c, (col, v) in enumerate(((W - 1, np.inf), (W - 2, -np.inf), (0, np.nan), (W - 1, np.nan))[:max(1, C - 1)]):
            x[(c + 1) % B, c, H // 2 + c, col] = v
    else:              # a filter each: the ends of a row, and the first column, which lies behind the row above
        for f, (col, v) in enumerate(((ow - 1, np.inf), (0, np.nan), (0, -np.inf))):
            dy[(f + 1) % B, f, oh // 2, col] = v
    _compare(ctx, x, dy, (pad, pad), code)


# B, C, H, W, F, padH, padW: up to six values in an image, rows made of padding
TINY = [(40, 1, 1, 2, 8, 1, 5), (40, 2, 1, 2, 8, 1, 5), (40, 1, 2, 2, 9, 1, 6), (40, 1, 1, 3, 16, 1, 5), (60, 3, 1, 1, 8, 1, 5),
        (60, 4, 1, 1, 8, 1, 8), (40, 1, 1, 5, 8, 1, 4), (40, 1, 2, 3, 8, 1, 5), (40, 5, 1, 1, 8, 1, 6), (30, 1, 2, 1, 8, 3, 7)]


@pytest.mark.parametrize("dt", ["f32", "f64"])
@pytest.mark.parametrize("cfg", TINY)
def test_images_of_a_few_values(ctx, cfg, dt):
    np_dt, code = (np.float32, _ffi.F32) if dt == "f32" else (np.float64, _ffi.F64)
    B, C, H, W, F, padH, padW = cfg
    oh, ow = H + 2 * padH - 2, W + 2 * padW - 2
    if dt == "f32":   # enough pixels for the matrix-core kernel
        B = -(-70000 // (oh * ow))
    rng = np.random.default_rng(B + W)
    x = rng.uniform(-1, 1, (B, C, H, W)).astype(np_dt)
    dy = rng.uniform(-1, 1, (B, F, oh, ow)).astype(np_dt)
    _compare(ctx, x, dy, (padH, padW), code)
