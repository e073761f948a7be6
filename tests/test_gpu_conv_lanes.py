"""k_conv3x3_lanes: 3x3 stride-1 convolutions and image gradients with operands straight from memory, at the edges of
their pixel groups, tiles and forms, against float64 sums over shifted images; and the kernels it stands in for."""
from ctypes import byref as C_byref

import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests import test_gpu_nn as NN
from tests.util import assert_bits_equal, rel_frobenius

pytestmark = pytest.mark.gpu

# B, C, H, W, F, padH: rows of one group, of one more column than groups, of 1 to 3 more; one quad per wavefront, fewer,
# more, an odd number; filters short of a tile; no, one and two rows of padding; two output rows; several tiles
CASES = [(1, 64, 26, 26, 128, 1), (1, 8, 30, 4, 16, 1), (2, 12, 21, 5, 17, 1), (1, 40, 17, 18, 33, 0), (3, 36, 9, 19, 8, 2),
         (1, 128, 13, 13, 100, 1), (2, 16, 52, 52, 32, 1), (1, 64, 52, 52, 64, 1), (1, 20, 4, 33, 24, 0), (8, 32, 52, 52, 64, 1),
         (3, 64, 7, 7, 130, 1), (1, 264, 10, 10, 48, 1)]
F64_CASES = CASES[:6] + [(50, 32, 14, 14, 64, 1), (256, 32, 14, 14, 64, 1), (20, 64, 7, 7, 128, 1)]


def _forward(x, w, padH):
    B, C, H, W = x.shape
    xp = np.zeros((B, C, H + 2 * padH, W + 2))
    xp[:, :, padH:padH + H, 1:1 + W] = x
    oh = H + 2 * padH - 2
    out = np.zeros((B, w.shape[0], oh, W))
    w = w.astype(np.float64)
    for ky in range(3):
        for kx in range(3):
            part = xp[:, :, ky:ky + oh, kx:kx + W].reshape(B, C, -1)
            out += np.matmul(w[:, :, ky, kx], part).reshape(out.shape)
    return out


def _run(ctx, cfg, dt, flip=False, **kw):
    B, C, H, W, F, padH = cfg
    np_dt, code = (np.float32, _ffi.F32) if dt == "f32" else (np.float64, _ffi.F64)
    rng = np.random.default_rng(sum(cfg) + flip)
    oh = H + 2 * padH - 2
    x = rng.standard_normal((B, F, oh, W) if flip else (B, C, H, W)).astype(np_dt)
    w = rng.standard_normal((F, C, 3, 3)).astype(np_dt)
    shape = (B, C, H, W) if flip else (B, F, oh // 2, W // 2) if kw.get("pool2") else (B, F, oh, W)
    bn = kw.pop("bn", None)
    px, pw, py = ctx.upload(x), ctx.upload(w), ctx.upload(np.full(shape, np.nan, np_dt))
    pbn = [ctx.upload(v) for v in bn] if bn else []
    if flip:
        ctx.run(D.cmd_conv2d_bwd_data(px, pw, py, B, C, H, W, F, 3, 3, (padH, 1), dtype=code))
    else:
        ctx.run(D.cmd_conv2d(px, pw, py, B, C, H, W, F, 3, 3, (padH, 1), dtype=code, bn=pbn or None, **kw))
    got = ctx.d2h(py, shape, np_dt)
    for p in [px, pw, py] + pbn:
        ctx.free(p)
    return x, w, got


@pytest.mark.parametrize("dt,cfg", [("f32", c) for c in CASES] + [("f64", c) for c in F64_CASES])
def test_forward_and_gradient(ctx, dt, cfg):
    bar = 2e-6 if dt == "f32" else 1e-14   # sums of at most 9 x 264 products in the operands' own precision
    x, w, got = _run(ctx, cfg, dt)
    assert rel_frobenius(got, _forward(x, w, cfg[5])) <= bar
    if cfg[4] % 4 == 0 and cfg[5] <= 2:
        dy, w, got = _run(ctx, cfg, dt, flip=True)
        mirrored = w[:, :, ::-1, ::-1].transpose(1, 0, 2, 3)
        assert rel_frobenius(got, _forward(dy, mirrored, 2 - cfg[5])) <= bar


@pytest.mark.parametrize("cfg", [c for c in CASES if c[2] + 2 * c[5] - 2 >= 2])
def test_epilogues_on_the_plain_result(ctx, cfg):
    """Activation and pooling, alone and together, are those of the plain result bit for bit."""
    _, _, z = _run(ctx, cfg, "f32")
    F, oh, ow = z.shape[1:]
    _, _, got = _run(ctx, cfg, "f32", act="relu")
    a = z * (z >= 0)
    assert_bits_equal(got, a, "rectified")
    B, C, H, W, _, padH = cfg
    if not ctx.lib.gh_conv2d_can_pool(C_byref(D.cmd_conv2d(0x1000, 0x2000, 0x3000, B, C, H, W, F, 3, 3, (padH, 1), pool2=True))):
        return
    pooled = a[:, :, :oh // 2 * 2, :ow // 2 * 2].reshape(B, F, oh // 2, 2, ow // 2, 2).max((3, 5))
    _, _, got = _run(ctx, cfg, "f32", act="relu", pool2=True)
    assert np.array_equal(got, pooled)
    rng = np.random.default_rng(9)
    bn = [rng.standard_normal(F).astype(np.float32), rng.uniform(0.5, 2, F).astype(np.float32),
          rng.standard_normal(F).astype(np.float32), rng.standard_normal(F).astype(np.float32)]
    scale = np.float32(1) / np.sqrt(bn[1] + np.float32(1e-5))
    v = z * scale[:, None, None] + (-bn[0] * scale)[:, None, None]
    v = bn[2][:, None, None] * v + bn[3][:, None, None]
    v = v * (v >= 0) + (v * (v < 0)) * np.float32(0.1)
    pooled = v[:, :, :oh // 2 * 2, :ow // 2 * 2].reshape(B, F, oh // 2, 2, ow // 2, 2).max((3, 5))
    _, _, got = _run(ctx, cfg, "f32", act="leaky", alpha=0.1, pool2=True, bn=bn)
    assert np.array_equal(got, pooled)


@pytest.mark.parametrize("cfg", NN.PATCH_CASES)
def test_patch_kernel_stays_right(ctx, monkeypatch, cfg):
    monkeypatch.setenv("GORGONIA_HIP_CONV_NO_LANES", "1")
    NN.test_conv_patch_kernel(ctx, cfg)


@pytest.mark.parametrize("cfg", NN.WIDE_CASES[:6])
def test_wide_kernel_stays_right(ctx, monkeypatch, cfg):
    monkeypatch.setenv("GORGONIA_HIP_CONV_NO_LANES", "1")
    NN.test_conv_wide_kernel(ctx, cfg)
