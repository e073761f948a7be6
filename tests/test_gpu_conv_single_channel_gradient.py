"""The filter gradient over single-channel images (k_conv3x3_wgrad_c1): images fetched ahead and larger ones, whole and partial
groups of pixels, more images than workgroups and fewer, filters past a workgroup's four, infinities and NaN in the last pixel's
window and in the last pixel, which reach the taps that read them and no other."""
import numpy as np
import pytest
import torch

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.test_gpu_conv_filter_gradient_edges import _compare

pytestmark = pytest.mark.gpu

# B, H, W, F, pad
CASES = [(128, 28, 28, 32, 1), (200, 28, 28, 10, 1), (3, 30, 30, 5, 1), (130, 31, 29, 8, 1), (70, 32, 32, 9, 0), (65, 33, 33, 4, 0), (5, 110, 100, 6, 1), (129, 10, 9, 33, 1), (1, 8, 8, 32, 1),
         (70, 24, 24, 7, 0), (66, 64, 16, 3, 1)]


@pytest.mark.parametrize("B,H,W,F,pad", CASES)
def test_against_64_bit_sums(ctx, B, H, W, F, pad):
    oh, ow = H + 2 * pad - 2, W + 2 * pad - 2
    rng = np.random.default_rng(B + H * W)
    x, dy = rng.standard_normal((B, 1, H, W)).astype(np.float32), rng.standard_normal((B, F, oh, ow)).astype(np.float32)
    at = [ctx.upload(x), ctx.upload(dy), ctx.upload(np.full(F * 9 + 64, np.nan, np.float32))]
    cmd = D.cmd_conv2d_bwd_filter(at[0], at[1], at[2], B, 1, H, W, F, 3, 3, (pad, pad))
    results = []
    for _ in range(2):
        ctx.run([cmd])
        results.append(ctx.d2h(at[2], (F * 9 + 64,)))
    for p in at:
        ctx.free(p)
    got = results[0][:F * 9]
    assert np.array_equal(got.view(np.uint32), results[1][:F * 9].view(np.uint32)) and np.isnan(results[0][F * 9:]).all()
    want = torch.nn.grad.conv2d_weight(torch.from_numpy(x).double(), (F, 1, 3, 3), torch.from_numpy(dy).double(), padding=pad).numpy().ravel()
    # n products in lanes' sums of n / (64 workgroups' 64 lanes) at most and some twelve additions behind them: each rounds by
    # 2^-24 of a partial sum, which grows as the square root of its products
    chain = -(-B // 64) * -(-oh * ow // 64) + 12
    assert np.linalg.norm(got - want) <= np.sqrt(chain) * 2.0 ** -24 * np.linalg.norm(want)


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("where", ["x", "dy"])
@pytest.mark.parametrize("B,H,W,F,pad", CASES)
def test_infinities_and_nan_at_the_end_of_an_image(ctx, B, H, W, F, pad, where, value):
    rng = np.random.default_rng(B + W)
    x = rng.standard_normal((B, 1, H, W)).astype(np.float32)
    dy = rng.standard_normal((B, F, H + 2 * pad - 2, W + 2 * pad - 2)).astype(np.float32)
    if where == "x":
        x[B // 2, 0, -1, -1] = value
    else:
        dy[B // 2, F // 2, -1, -1] = value
    _compare(ctx, x, dy, (pad, pad), _ffi.F32)
