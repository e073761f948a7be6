"""The training statistics of BatchNorm from partial sums per workgroup: groups at the edges of strips and images,
and values whose mean is large against their spread, against float64."""
import numpy as np
import pytest

from gorgonia_amd import device as D

pytestmark = pytest.mark.gpu


# planes of one strip, of one column more and less than strips, narrow planes over many images, one image, offsets
@pytest.mark.parametrize("B,C,S,offset", [(8, 3, 256, 0), (5, 4, 257, 1), (3, 2, 1023, 100), (9, 5, 2600, 3), (7, 3, 255, 10), (4100, 6, 1, 2),
                                          (2500, 3, 9, 50), (1, 7, 4000, 1000), (2, 2, 43264, 1000), (6, 16, 10816, 0.5)])
def test_statistics(ctx, B, C, S, offset):
    rng = np.random.default_rng(B + S)
    x = (rng.standard_normal((B, C, S)) * rng.uniform(0.5, 3, (1, C, 1)) + offset).astype(np.float32)
    rm0, rv0 = rng.standard_normal(C).astype(np.float32), rng.uniform(1, 2, C).astype(np.float32)
    px, py = ctx.upload(x), ctx.malloc(x.nbytes)
    stats = [ctx.upload(v) for v in (rm0, rv0, np.zeros(C, np.float32), np.zeros(C, np.float32))]
    ctx.run(D.cmd_bn_train(px, py, *stats, B, C, S, 1e-5, 0.9))
    y = ctx.d2h(py, x.shape, np.float32)
    rm, rv, sm, sv = (ctx.d2h(p, (C,), np.float32) for p in stats)
    for p in [px, py] + stats:
        ctx.free(p)
    n = B * S
    x64 = x.astype(np.float64)
    mean = x64.mean((0, 2))
    dev = ((x64 - mean[None, :, None]) ** 2).sum((0, 2))
    # a sum's tree of at most some 200 steps, each rounding by 2^-24 of the partial sum
    assert np.allclose(sm, mean, rtol=2e-6, atol=2e-6)
    assert np.allclose(sv, dev, rtol=5e-6)
    assert np.allclose(rm, 0.9 * mean + 0.1 * rm0, rtol=3e-6, atol=3e-6)
    assert np.allclose(rv, 0.9 * dev / (n - 1) + 0.1 * rv0, rtol=1e-5)
    want = (x64 - mean[None, :, None]) / np.sqrt(dev / n + 1e-5)[None, :, None]
    # x a - mean a: two roundings of the size of the offset
    assert np.abs(y - want).max() <= 1e-5 + 4e-7 * abs(offset) / 0.5 * 4
