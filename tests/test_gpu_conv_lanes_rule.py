"""3x3 convolutions and image gradients that k_conv3x3_lanes takes from the patch kernel: against 64-bit sums, and the pooled
result against the plain one's."""
import ctypes as C

import numpy as np
import pytest
import torch

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.util import assert_bits_equal

# a sum of n products in float32 is off by about sqrt(n) 2^-25 of the norm of normal values' results; chains of n / 8 and seven
# additions stay below half of that
def _bound(n):
    return 0.5 * np.sqrt(n) * 2.0 ** -25


# B, C, H, W, F
FORWARD = [(7, 512, 8, 8, 1024), (5, 256, 9, 9, 512), (3, 192, 9, 7, 128), (1, 192, 24, 21, 32), (4, 96, 47, 39, 64), (2, 192, 21, 21, 512), (1, 64, 52, 52, 128), (1, 128, 26, 26, 256)]
GRADIENT = [(8, 32, 52, 52, 64), (13, 64, 40, 49, 64), (18, 64, 23, 22, 256), (2, 128, 90, 86, 64)]


def _straight(cmd):
    return _ffi.load().gh_runs_straight(C.byref(cmd))


def test_route():
    for B, Cn, H, W, F in FORWARD:
        assert _straight(D.cmd_conv2d(0x10000, 0x20000, 0x30000, B, Cn, H, W, F, 3, 3, (1, 1))) == 1, (B, Cn, H, W, F)
    for B, Cn, H, W, F in GRADIENT:
        assert _straight(D.cmd_conv2d_bwd_data(0x10000, 0x20000, 0x30000, B, Cn, H, W, F, 3, 3, (1, 1))) == 1, (B, Cn, H, W, F)
    # the patch kernel's still: shapes for which the eight wavefronts' form is no quicker
    for B, Cn, H, W, F in ((8, 512, 13, 13, 1024), (8, 64, 26, 26, 128), (8, 256, 13, 13, 512)):
        assert _straight(D.cmd_conv2d(0x10000, 0x20000, 0x30000, B, Cn, H, W, F, 3, 3, (1, 1))) == 0, (B, Cn, H, W, F)


@pytest.mark.gpu
@pytest.mark.parametrize("B,Cn,H,W,F", FORWARD)
def test_forward(ctx, B, Cn, H, W, F):
    rng = np.random.default_rng(B * Cn + H)
    x, w = rng.standard_normal((B, Cn, H, W)).astype(np.float32), rng.standard_normal((F, Cn, 3, 3)).astype(np.float32)
    at = [ctx.upload(x), ctx.upload(w), ctx.upload(np.full((B, F, H, W), np.nan, np.float32)), ctx.upload(np.full((B, F, H // 2, W // 2), np.nan, np.float32))]
    plain = D.cmd_conv2d(at[0], at[1], at[2], B, Cn, H, W, F, 3, 3, (1, 1))
    ctx.run([plain])
    got = ctx.d2h(at[2], (B, F, H, W))
    want = torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(w).double(), padding=1).numpy()
    assert np.linalg.norm(got - want) <= _bound(9 * Cn) * np.linalg.norm(want)
    pooled = D.cmd_conv2d(at[0], at[1], at[3], B, Cn, H, W, F, 3, 3, (1, 1), pool2=True)
    can = _ffi.load().gh_conv2d_can_pool(C.byref(plain))
    assert can or Cn < 64
    if can:
        ctx.run([pooled])
        assert_bits_equal(ctx.d2h(at[3], (B, F, H // 2, W // 2)), got[:, :, :H // 2 * 2, :W // 2 * 2].reshape(B, F, H // 2, 2, W // 2, 2).max(axis=(3, 5)))
    for p in at:
        ctx.free(p)


@pytest.mark.gpu
@pytest.mark.parametrize("units", [8, 32, 64, 104, 152, 208])
def test_pooled_with_other_numbers_of_compute_units(monkeypatch, units):
    """What gh_conv2d_can_pool accepts, for whatever number of compute units it answers, runs on a device with another number,
    and has the plain result's bits there too."""
    monkeypatch.setenv("GORGONIA_HIP_COMPUTE_UNITS", str(units))
    rng = np.random.default_rng(units)
    with D.Context() as ctx:
        for B, Cn, H, W, F in FORWARD:
            x, w = rng.standard_normal((B, Cn, H, W)).astype(np.float32), rng.standard_normal((F, Cn, 3, 3)).astype(np.float32)
            at = [ctx.upload(x), ctx.upload(w), ctx.upload(np.full((B, F, H, W), np.nan, np.float32)), ctx.upload(np.full((B, F, H // 2, W // 2), np.nan, np.float32))]
            plain = D.cmd_conv2d(at[0], at[1], at[2], B, Cn, H, W, F, 3, 3, (1, 1))
            if _ffi.load().gh_conv2d_can_pool(C.byref(plain)):
                ctx.run([plain, D.cmd_conv2d(at[0], at[1], at[3], B, Cn, H, W, F, 3, 3, (1, 1), pool2=True)])
                got = ctx.d2h(at[2], (B, F, H, W))
                want = got[:, :, :H // 2 * 2, :W // 2 * 2].reshape(B, F, H // 2, 2, W // 2, 2).max(axis=(3, 5))
                assert_bits_equal(ctx.d2h(at[3], (B, F, H // 2, W // 2)), want)
            for p in at:
                ctx.free(p)


@pytest.mark.gpu
@pytest.mark.parametrize("B,Cn,H,W,F", GRADIENT)
def test_gradient(ctx, B, Cn, H, W, F):
    rng = np.random.default_rng(B * Cn + H)
    dy, w = rng.standard_normal((B, F, H, W)).astype(np.float32), rng.standard_normal((F, Cn, 3, 3)).astype(np.float32)
    at = [ctx.upload(dy), ctx.upload(w), ctx.upload(np.full((B, Cn, H, W), np.nan, np.float32))]
    ctx.run([D.cmd_conv2d_bwd_data(at[0], at[1], at[2], B, Cn, H, W, F, 3, 3, (1, 1))])
    got = ctx.d2h(at[2], (B, Cn, H, W))
    want = torch.nn.functional.conv_transpose2d(torch.from_numpy(dy).double(), torch.from_numpy(w).double(), padding=1).numpy()
    assert np.linalg.norm(got - want) <= _bound(9 * F) * np.linalg.norm(want)
    for p in at:
        ctx.free(p)
