"""k_gemm_split: float32 products on the bf16 matrix instructions, values split into three bf16 parts.  Every form
at edges of its tiles, steps and parts of K, transposes, leading dimensions, operands that are only 4-byte aligned, batches,
epilogues, and the values the split cannot hold (infinities, NaN, the largest), against float64 products."""
import ctypes as C

import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.util import rel_frobenius

pytestmark = pytest.mark.gpu

# 128 x 128; the same in two parts of K; 64 x 64 in two parts; in four
SHAPES = [(3800, 4001, 131, 1), (640, 650, 18, 40), (2047, 2049, 95, 1), (2000, 2000, 47, 1), (2176, 1900, 64, 1), (1025, 1023, 129, 4),
          (255, 513, 97, 30), (1200, 2100, 333, 1), (500, 500, 500, 8), (1000, 1000, 1025, 1), (1024, 1024, 1024, 1)]


def _cmd(pa, pb, pc, m, n, k, batch, **kw):
    cmd = D.cmd_gemm(pa, pb, pc, m, n, k, batch=batch, **kw)
    assert _ffi.load().gh_runs_split(C.byref(cmd)) == 1, (m, n, k, batch)
    return cmd


def _run(ctx, a, b, m, n, k, batch=1, ta=False, tb=False, pad=0, shift=0, **kw):
    """a, b: what lies in memory, (batch, rows, columns + pad); shift: floats in front of each tensor."""
    front = np.full(shift, np.nan, np.float32)
    held = [ctx.upload(np.concatenate([front, t.ravel()]) if shift else t) for t in (a, b)]
    pc = ctx.upload(np.full(batch * m * (n + pad) + shift, np.nan, np.float32))
    o = 4 * shift
    ctx.run(_cmd(held[0] + o, held[1] + o, pc + o, m, n, k, batch, trans_a=ta, trans_b=tb, lda=a.shape[2], ldb=b.shape[2], ldc=n + pad,
                 stride_a=a[0].size, stride_b=b[0].size, stride_c=m * (n + pad), **kw))
    got = ctx.d2h(pc + o, (batch, m, n + pad))
    for p in held + [pc]:
        ctx.free(p)
    assert pad == 0 or np.isnan(got[:, :, n:]).all()   # nothing is stored past the columns
    return got[:, :, :n]


def _inputs(m, n, k, batch, ta, tb, pad=0, seed=0):
    rng = np.random.default_rng(m * 7 + n * 3 + k + batch + seed)
    a = rng.standard_normal((batch, k if ta else m, (m if ta else k) + pad), np.float32)
    b = rng.standard_normal((batch, n if tb else k, (k if tb else n) + pad), np.float32)
    x, y = a[:, :, :a.shape[2] - pad].astype(np.float64), b[:, :, :b.shape[2] - pad].astype(np.float64)
    return a, b, (x.transpose(0, 2, 1) if ta else x), (y.transpose(0, 2, 1) if tb else y)


# 16 k are summed exactly but for one rounding of the sum, 2^-24 of its size at most, a third of that on average, and the roundings
# add up as their root: K = 1025 gives sqrt(65) * 2^-24 / sqrt(3) * sqrt(1/2) = 2.0e-7.
@pytest.mark.parametrize("m,n,k,batch", SHAPES)
def test_product(ctx, m, n, k, batch):
    for ta, tb in ((False, False), (True, False), (False, True), (True, True)):
        a, b, x, y = _inputs(m, n, k, batch, ta, tb)
        assert rel_frobenius(_run(ctx, a, b, m, n, k, batch, ta, tb), np.matmul(x, y)) <= 3e-7, (ta, tb)


@pytest.mark.parametrize("m,n,k,batch", [(2176, 1900, 64, 1), (500, 500, 500, 8)])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
def test_wider_leading_dimensions_at_any_float(ctx, m, n, k, batch, ta, tb):
    a, b, x, y = _inputs(m, n, k, batch, ta, tb, pad=3)
    assert rel_frobenius(_run(ctx, a, b, m, n, k, batch, ta, tb, pad=3, shift=1), np.matmul(x, y)) <= 3e-7


# 0.5 for rounding the sum, and of the seven smaller products, 2^-7 of the first, three roundings of half their last place at most
@pytest.mark.parametrize("m,n,k,batch", [(2000, 2000, 47, 1), (1200, 2100, 333, 1), (500, 500, 500, 8), (1024, 1024, 1024, 1)])
def test_one_product_to_a_result(ctx, m, n, k, batch):
    rng = np.random.default_rng(m + k)
    a, b = np.zeros((batch, m, k), np.float32), rng.standard_normal((batch, k, n), np.float32)
    at = rng.integers(0, k, (batch, m))
    scale = rng.standard_normal((batch, m), np.float32)
    np.put_along_axis(a, at[:, :, None], scale[:, :, None], 2)
    want = scale[:, :, None].astype(np.float64) * np.take_along_axis(b, np.repeat(at[:, :, None], n, 2), 1)
    last = np.spacing(np.abs(want).astype(np.float32)).astype(np.float64)
    assert (np.abs(_run(ctx, a, b, m, n, k, batch) - want) / last).max() <= 0.5 + 1.5 / 128


@pytest.mark.parametrize("m,n,k", [(4096, 4096, 4096), (2048, 2048, 2048), (2321, 3480, 2049), (2649, 3563, 3143), (1000, 1000, 4000)])
@pytest.mark.parametrize("values", ["normal", "uniform"])
def test_error_is_no_larger_than_on_the_float32_instructions(ctx, monkeypatch, m, n, k, values):
    rng = np.random.default_rng(k)
    a, b = (rng.standard_normal(s, np.float32) if values == "normal" else rng.random(s, np.float32) for s in ((1, m, k), (1, k, n)))
    want = np.matmul(a[0].astype(np.float64), b[0].astype(np.float64))
    split = rel_frobenius(_run(ctx, a, b, m, n, k)[0], want)
    monkeypatch.setitem(globals(), "_cmd", lambda pa, pb, pc, m, n, k, batch, **kw: D.cmd_gemm(pa, pb, pc, m, n, k, batch=batch, **kw))
    monkeypatch.setenv("GORGONIA_HIP_NO_SPLIT", "1")
    assert split <= rel_frobenius(_run(ctx, a, b, m, n, k)[0], want)


def test_whole_numbers_are_exact(ctx):
    rng = np.random.default_rng(3)
    a, b = (rng.integers(-60, 61, s).astype(np.float32) for s in ((1, 1024, 1024), (1, 1024, 1024)))
    assert np.array_equal(_run(ctx, a, b, 1024, 1024, 1024), np.matmul(a.astype(np.float64), b.astype(np.float64)))


def test_bias_and_activation(ctx):
    m, n, k = 2000, 2000, 47
    a, b, _, _ = _inputs(m, n, k, 1, False, False)
    bias = np.random.default_rng(1).standard_normal(n, np.float32)
    bare, pb = _run(ctx, a, b, m, n, k), ctx.upload(bias)
    z = bare + bias
    assert np.array_equal(_run(ctx, a, b, m, n, k, bias=pb, act="relu"), z * (z >= 0))
    assert np.array_equal(_run(ctx, a, b, m, n, k, act="leaky", alpha=0.1), bare * (bare >= 0) + (bare * (bare < 0)) * np.float32(0.1))
    ctx.free(pb)


@pytest.mark.parametrize("m,n,k,batch", [(640, 650, 18, 40), (500, 500, 500, 8)])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)])
def test_values_the_split_cannot_hold(ctx, m, n, k, batch, ta, tb):
    """Infinities, NaN, values and sums that only float32 itself can hold: their tiles come from the float32 instructions."""
    a, b, x, y = _inputs(m, n, k, batch, ta, tb)
    x, y = np.ascontiguousarray(x), np.ascontiguousarray(y)
    x[0, 3, 1], x[1, m - 1, k - 1], y[1, 2, 77] = np.inf, np.nan, -np.inf
    x[2, 40], y[2, :, 9] = 2e38 / k, 1.0        # a row of the largest values, a column that keeps their sum in range
    y[3, :, n - 1] *= np.float32(1e30)
    x, y = x.astype(np.float32), y.astype(np.float32)
    a = np.ascontiguousarray(x.transpose(0, 2, 1) if ta else x)
    b = np.ascontiguousarray(y.transpose(0, 2, 1) if tb else y)
    got = _run(ctx, a, b, m, n, k, batch, ta, tb)
    with np.errstate(invalid="ignore", over="ignore"):
        want = np.matmul(x.astype(np.float64), y.astype(np.float64))
        # a sum beyond float32 is an infinity wherever its partial sums overflow, which is a matter of order: left out near the limit
        sure = ~(np.abs(want) > 1e38) | np.isinf(want)
        sure[2, 40] = False
        sure[2, 40, 9] = True
        want32 = want.astype(np.float32)
        assert np.array_equal(np.isnan(got[sure]), np.isnan(want32[sure]))
        assert np.array_equal(np.where(np.isinf(got), got, 0)[sure], np.where(np.isinf(want32), want32, 0)[sure])
    fin = sure & np.isfinite(want32)
    assert abs(got[2, 40, 9] / want[2, 40, 9] - 1) <= 1e-6
    for z in range(4):
        for cols in (slice(0, n - 1), slice(n - 1, n)):
            f = fin[z, :, cols].copy()
            f[40] &= z != 2
            assert rel_frobenius(got[z, :, cols][f], want[z, :, cols][f]) <= 1e-6


# the places where a workgroup looks at its sums: early, on the way (from 560 k in one part) and at the end
@pytest.mark.parametrize("m,n,k,batch", [(640, 650, 18, 40), (3000, 3001, 700, 1), (1200, 2100, 333, 1), (500, 500, 500, 8), (1024, 1024, 1024, 1)])
@pytest.mark.parametrize("place", [0.0, 0.6, 1.0])
@pytest.mark.parametrize("value", [np.nan, np.inf, -3.4e38])
def test_one_value_that_the_split_cannot_hold(ctx, m, n, k, batch, place, value):
    a, b, x, y = _inputs(m, n, k, batch, False, False)
    row, at = m - 2, int(place * (k - 1))
    a[batch - 1, row, at] = value
    b[:, at] = np.where(np.abs(b[:, at]) > 0.5, 0.5, b[:, at])   # (a product of the largest value stays a float32)
    got = _run(ctx, a, b, m, n, k, batch)
    want = np.matmul(a.astype(np.float64), b.astype(np.float64)) if np.isfinite(value) else None
    if want is None:
        bad = np.float32(value) * b[batch - 1, at]
        assert np.array_equal(got[batch - 1, row], bad, equal_nan=True)
        a[batch - 1, row] = 0.0
        want = np.matmul(a.astype(np.float64), b.astype(np.float64))
        got[batch - 1, row] = 0.0
    else:
        assert rel_frobenius(got[batch - 1, row], want[batch - 1, row]) <= 1e-6
        got[batch - 1, row] = want[batch - 1, row] = 0.0
    assert rel_frobenius(got, want) <= 3e-7


# A tile that is computed twice takes both kernels' times (less than twice the slower one's), and some more where a compute
# unit has one tile.
@pytest.mark.parametrize("m,n,k,batch", [(2048, 2048, 2048, 1), (1024, 1024, 1024, 1), (512, 512, 512, 64)])
def test_time_of_values_that_the_split_cannot_hold(ctx, monkeypatch, m, n, k, batch):
    a = np.full((batch, m, k), np.nan, np.float32)
    p = [ctx.upload(a), ctx.upload(a), ctx.malloc(4 * batch * m * n)]
    cmd = _cmd(*p, m, n, k, batch, stride_a=m * k, stride_b=k * n, stride_c=m * n)

    def ms():
        ctx.run([cmd] * 20)
        ctx.event(0)
        ctx.submit([cmd] * 20)
        ctx.event(1)
        return ctx.elapsed_ms(0, 1)
    split = min(ms() for _ in range(5))
    monkeypatch.setenv("GORGONIA_HIP_NO_SPLIT", "1")
    assert split <= 3 * min(ms() for _ in range(5))
    for q in p:
        ctx.free(q)


@pytest.mark.parametrize("scale", [1e-30, 1e-36, 1e-39])
def test_small_and_denormal_values_keep_their_bits(ctx, scale):
    m, n, k = 1024, 1024, 1024
    a, b, _, _ = _inputs(m, n, k, 1, False, False)
    a = (a.astype(np.float64) * scale).astype(np.float32)
    want = np.matmul(a.astype(np.float64), b.astype(np.float64))
    # results below 2^-126 are rounded to multiples of 2^-149
    assert np.abs(_run(ctx, a, b, m, n, k) - want).max() <= 2e-6 * np.abs(want).max() + 2.0 ** -149
