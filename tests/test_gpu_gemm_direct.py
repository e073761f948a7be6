"""k_gemm_direct: products with operands straight from memory.  Every form, transpose and edge of its tiles, groups
and chunks, leading dimensions wider than the matrix, batches, and the epilogues, against float64 products."""
import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.util import rel_frobenius

pytestmark = pytest.mark.gpu

# m, n, k, batch: forms by size; one row or column more or less than tiles of 32, 48, 64, 80 and 128; k of whole chunks,
# one more, one less, less than one chunk, and around the chunk pairs of four and eight wavefronts
SHAPES = [(333, 900, 300, 1), (640, 640, 257, 1), (641, 639, 255, 1), (1000, 513, 129, 1), (1201, 331, 127, 1), (777, 1543, 61, 1),
          (5, 4, 17, 300), (33, 65, 16, 70), (81, 127, 15, 33), (47, 63, 1, 129), (129, 70, 200, 40), (320, 1300, 1100, 1),
          (1153, 625, 513, 1), (80, 64, 31, 64), (700, 1030, 96, 1), (4, 5000, 40, 4)]


@pytest.fixture(scope="module")
def ctx():
    c = D.Context(0, 0)
    yield c
    c.close()


def _case(ctx, m, n, k, batch, ta, tb, dt, pad=0, bias=None, act=None):
    np_dt, code = (np.float32, _ffi.F32) if dt == "f32" else (np.float64, _ffi.F64)
    rng = np.random.default_rng(m * 7 + n * 3 + k + batch)
    sa, sb = ((k, m) if ta else (m, k)), ((n, k) if tb else (k, n))
    a = rng.standard_normal((batch, sa[0], sa[1] + pad)).astype(np_dt)
    b = rng.standard_normal((batch, sb[0], sb[1] + pad)).astype(np_dt)
    pa, pb, pc = ctx.upload(a), ctx.upload(b), ctx.upload(np.full((batch, m, n + pad), np.nan, np_dt))
    pbias = ctx.upload(bias) if bias is not None else 0
    ctx.run(D.cmd_gemm(pa, pb, pc, m, n, k, lda=sa[1] + pad, ldb=sb[1] + pad, ldc=n + pad, trans_a=ta, trans_b=tb, batch=batch,
                       stride_a=a[0].size, stride_b=b[0].size, stride_c=m * (n + pad), dtype=code, bias=pbias, act=act, alpha=0.1))
    got = ctx.d2h(pc, (batch, m, n + pad), np_dt)
    for p in (pa, pb, pc) + ((pbias,) if pbias else ()):
        ctx.free(p)
    x, y = a[:, :, :sa[1]].astype(np.float64), b[:, :, :sb[1]].astype(np.float64)
    want = np.matmul(x.transpose(0, 2, 1) if ta else x, y.transpose(0, 2, 1) if tb else y)
    assert pad == 0 or np.isnan(got[:, :, n:]).all()   # nothing is stored past the columns
    return got[:, :, :n], want



# float64 products of one tile to a compute unit: eight wavefronts from K = 640 on, with whole pairs of chunks for each, one chunk
# more, one less and a last one that is short
@pytest.mark.parametrize("m,n,k", [(113, 1444, 1480), (370, 661, 860), (777, 1543, 641), (320, 1300, 1024), (31, 30, 648), (64, 900, 639)])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
def test_float64_in_eight_slices(ctx, m, n, k, ta, tb):
    got, want = _case(ctx, m, n, k, 1, ta, tb, "f64")[:2]
    assert rel_frobenius(got, want) <= 1e-15 * np.sqrt(k / 8) + 2.0 ** -53 * 8   # a slice's roundings as their root, and eight sums


@pytest.mark.parametrize("dt,bar", [("f32", 1e-5), ("f64", 1e-14)])
@pytest.mark.parametrize("m,n,k,batch", SHAPES)
def test_product(ctx, m, n, k, batch, dt, bar):
    for ta in (False, True):
        for tb in (False, True):
            got, want = _case(ctx, m, n, k, batch, ta, tb, dt)
            assert rel_frobenius(got, want) <= bar, (ta, tb)


@pytest.mark.parametrize("dt,bar", [("f32", 1e-5), ("f64", 1e-14)])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
def test_wider_leading_dimensions(ctx, ta, tb, dt, bar):
    got, want = _case(ctx, 515, 390, 145, 1, ta, tb, dt, pad=3)
    assert rel_frobenius(got, want) <= bar


@pytest.mark.parametrize("m,n,k", [(333, 900, 300), (1201, 331, 127)])
def test_bias_and_activation(ctx, m, n, k):
    bias = np.random.default_rng(1).standard_normal(n).astype(np.float32)
    bare, _ = _case(ctx, m, n, k, 1, False, False, "f32")
    got, _ = _case(ctx, m, n, k, 1, False, False, "f32", bias=bias, act="relu")
    z = bare + bias
    assert np.array_equal(got, z * (z >= 0))
    got, _ = _case(ctx, m, n, k, 1, False, False, "f32", act="leaky")
    assert np.array_equal(got, bare * (bare >= 0) + (bare * (bare < 0)) * np.float32(0.1))


@pytest.mark.parametrize("m,n,k,batch", [(1, 300, 40, 3), (300, 1, 40, 3), (1, 1, 5, 7), (1, 5, 1, 1)])
def test_rows_and_columns_of_one(ctx, m, n, k, batch):
    for dt, bar in (("f32", 1e-5), ("f64", 1e-14)):
        for ta, tb in ((False, False), (True, False), (False, True), (True, True)):
            got, want = _case(ctx, m, n, k, batch, ta, tb, dt)
            assert rel_frobenius(got, want) <= bar, (dt, ta, tb)
