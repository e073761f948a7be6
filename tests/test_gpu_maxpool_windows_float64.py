"""The float64 gradient of a 2x2 stride-2 pooling, a thread per window: odd and even extents, the smallest, tensors that
do not start on 16 bytes, ties, NaN and the type's lowest value, bit for bit against the oracle."""
import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from oracle import binding as O
from tests.util import assert_bits_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("B,C,H,W", [(1, 1, 2, 2), (2, 3, 2, 3), (2, 3, 3, 2), (1, 2, 5, 7), (3, 2, 28, 28), (2, 4, 7, 8), (2, 40, 33, 64)])
def test_windows(ctx, B, C, H, W, offset):
    rng = np.random.default_rng(H * W)
    x = rng.integers(-3, 4, (B, C, H, W)).astype(np.float64)   # many ties
    x[rng.random(x.shape) < 0.1] = np.nan
    x[rng.random(x.shape) < 0.2] = -np.finfo(np.float64).max
    dy = rng.standard_normal((B, C, H // 2, W // 2))
    want = O.maxpool2d_bwd(x, dy, (2, 2), (0, 0), (2, 2))
    pad = np.zeros(offset)
    px, py = ctx.upload(np.concatenate([pad, x.ravel()])), ctx.upload(np.concatenate([pad, dy.ravel()]))
    pd = ctx.upload(np.full(x.size + offset, np.nan))
    ctx.run(D.cmd_maxpool2d_bwd(px + 8 * offset, py + 8 * offset, pd + 8 * offset, B, C, H, W, 2, 2, (0, 0), (2, 2), dtype=_ffi.F64))
    got = ctx.d2h(pd, (x.size + offset,), np.float64)[offset:].reshape(x.shape)
    for p in (px, py, pd):
        ctx.free(p)
    assert_bits_equal(got, want, "pooling gradient")
