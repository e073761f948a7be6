"""k_gemm_thin: products of one to four rows (and more, which it leaves), at the edges of its column groups, rounds of K and row counts, against
float64 products."""
import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.util import rel_frobenius

pytestmark = pytest.mark.gpu


# columns: one more than a softmax's 32, one to three past a group and past a tile; K: a row per lane and fewer, one
# more and one less than a round of 128, several rounds, one more than eight of them
@pytest.mark.parametrize("n,k", [(33, 64), (48, 127), (49, 128), (300, 784), (301, 129), (302, 1025), (303, 1023), (100, 300), (4099, 513)])
@pytest.mark.parametrize("dt", ["f32", "f64"])
def test_thin_product(ctx, n, k, dt):
    np_dt, code, bar = (np.float32, _ffi.F32, 1e-6) if dt == "f32" else (np.float64, _ffi.F64, 2e-15)   # sqrt(K) roundings
    rng = np.random.default_rng(n + k)
    for m, pad in ((1, 0), (2, 3), (3, 1), (4, 0), (5, 2), (8, 5)):
        a, b = rng.standard_normal((m, k + pad)).astype(np_dt), rng.standard_normal((k, n + pad)).astype(np_dt)
        pa, pb, pc = ctx.upload(a), ctx.upload(b), ctx.upload(np.full((m, n + pad), np.nan, np_dt))
        kw = dict(lda=k + pad, ldb=n + pad, ldc=n + pad, dtype=code)
        ctx.run(D.cmd_gemm(pa, pb, pc, m, n, k, **kw))
        got = ctx.d2h(pc, (m, n + pad), np_dt)
        want = a[:, :k].astype(np.float64) @ b[:, :n].astype(np.float64)
        assert rel_frobenius(got[:, :n], want) <= bar, m
        assert pad == 0 or np.isnan(got[:, n:]).all()
        if dt == "f32":
            bias = rng.standard_normal(n).astype(np.float32)
            pbias = ctx.upload(bias)
            ctx.run(D.cmd_gemm(pa, pb, pc, m, n, k, bias=pbias, act="relu", **kw))
            z = got[:, :n] + bias
            assert np.array_equal(ctx.d2h(pc, (m, n + pad), np_dt)[:, :n], z * (z >= 0)), m
            ctx.free(pbias)
        for p in (pa, pb, pc):
            ctx.free(p)


def test_infinities_stay_in_their_columns(ctx):
    a, b = np.ones((2, 200), np.float32), np.ones((200, 50), np.float32)
    b[199, 7], b[3, 49], a[1, 199] = np.inf, -np.inf, 2
    pa, pb, pc = ctx.upload(a), ctx.upload(b), ctx.malloc(400)
    ctx.run(D.cmd_gemm(pa, pb, pc, 2, 50, 200))
    got = ctx.d2h(pc, (2, 50), np.float32)
    for p in (pa, pb, pc):
        ctx.free(p)
    assert np.array_equal(got, a @ b)
