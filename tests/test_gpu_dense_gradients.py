"""A dense layer's weight gradient and input gradient in one launch (k_gemm_gradients.hip): the bits of the two products
submitted apart, in both orders, and of what lies around their results."""
import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.util import assert_bits_equal

pytestmark = pytest.mark.gpu

# (batch, inputs, outputs): each kernel with each it stands beside, tiles that the sizes fill and do not, the smallest
# contractions, and products that one launch has no kernel for
F32 = [(128, 1152, 625), (128, 625, 10), (8, 1152, 625), (8, 625, 10), (31, 1152, 625), (33, 625, 10), (49, 1152, 625), (200, 1152, 625), (64, 784, 300),
       (64, 300, 100), (64, 100, 10), (37, 99, 41), (17, 530, 513), (16, 33, 600), (100, 47, 515), (5, 7, 9), (4, 16, 4), (300, 1152, 625), (2, 700, 10), (90, 2000, 30),
       (15, 400, 300), (9, 37, 333), (12, 2500, 140)]
F64 = [(50, 1152, 625), (50, 625, 10), (8, 1152, 625), (96, 1152, 625), (96, 625, 10), (13, 777, 300), (64, 300, 100), (100, 515, 77), (3, 5, 2), (70, 65, 260),
       (129, 31, 64), (64, 500, 3000), (40, 1600, 1600), (24, 2000, 2000), (2, 64, 3), (51, 778, 2019)]
CASES = [(np.float32,) + c for c in F32] + [(np.float64,) + c for c in F64]


def _commands(x, dy, w, dw, dx, batch, n_in, n_out, dtype, pad=0):
    return [D.cmd_gemm(x, dy, dw, n_in, n_out, batch, trans_a=True, ldc=n_out + pad, dtype=dtype),
            D.cmd_gemm(dy, w, dx, batch, n_in, n_out, trans_b=True, ldc=n_in + pad, dtype=dtype)]


@pytest.mark.parametrize("input_first", [False, True])
@pytest.mark.parametrize("dt,batch,n_in,n_out", CASES)
def test_both_gradients(ctx, dt, batch, n_in, n_out, input_first):
    rng = np.random.default_rng(batch * n_in + n_out)
    x = rng.standard_normal((batch, n_in)).astype(dt)
    dy = rng.standard_normal((batch, n_out)).astype(dt)
    w = rng.standard_normal((n_in, n_out)).astype(dt)
    dtype = _ffi.F64 if dt == np.float64 else _ffi.F32
    pad, edge = 3, 64
    dw_size, dx_size = n_in * (n_out + pad), batch * (n_in + pad)
    got = []
    for together in (True, False):
        at = [ctx.upload(a) for a in (x, dy, w)]
        dw, dx = (ctx.upload(np.full(n + 2 * edge, np.nan, dt)) for n in (dw_size, dx_size))
        off = edge * x.itemsize
        cmds = _commands(*at, dw + off, dx + off, batch, n_in, n_out, dtype, pad)
        if input_first:
            cmds.reverse()
        if together:
            ctx.run(cmds)
        else:
            for c in cmds:
                ctx.run([c])
        got.append([ctx.d2h(dw, (dw_size + 2 * edge,), dt), ctx.d2h(dx, (dx_size + 2 * edge,), dt)])
        for p in at + [dw, dx]:
            ctx.free(p)
    for a, b, rows in zip(*got, (n_in, batch)):
        assert_bits_equal(a, b)
        inside = a[edge:-edge].reshape(rows, -1)
        assert np.isnan(a[:edge]).all() and np.isnan(a[-edge:]).all() and np.isnan(inside[:, -pad:]).all() and not np.isnan(inside[:, :-pad]).any()


@pytest.mark.parametrize("which", ["x", "w"])
def test_result_that_the_other_reads(ctx, which):
    """An input gradient over the inputs that the weight gradient read, a weight gradient over the weights: as submitted apart."""
    batch, n_in, n_out = 128, 625, 10
    rng = np.random.default_rng(5)
    x, dy, w = (rng.standard_normal(s).astype(np.float32) for s in ((batch, n_in), (batch, n_out), (n_in, n_out)))
    got = []
    for together in (True, False):
        at = [ctx.upload(a) for a in (x, dy, w)]
        spare = ctx.upload(np.zeros_like(w if which == "x" else x))
        dw, dx = (spare, at[0]) if which == "x" else (at[2], spare)
        cmds = _commands(*at, dw, dx, batch, n_in, n_out, _ffi.F32)
        if together:
            ctx.run(cmds)
        else:
            for c in cmds:
                ctx.run([c])
        got.append([ctx.d2h(dw, w.shape), ctx.d2h(dx, x.shape)])
        for p in at + [spare]:
            ctx.free(p)
    for a, b in zip(*got):
        assert_bits_equal(a, b)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_operands_are_in_the_cache_account(dt):
    batch, n_in, n_out = 96, 625, 10
    rng = np.random.default_rng(7)
    with D.Context() as ctx:
        at = [ctx.upload(rng.standard_normal(s).astype(dt)) for s in ((batch, n_in), (batch, n_out), (n_in, n_out), (n_in, n_out), (batch, n_in))]
        assert not any(ctx.lib.gh_touched_lately(ctx.h, p) for p in at)
        ctx.run(_commands(*at, batch, n_in, n_out, _ffi.F64 if dt == np.float64 else _ffi.F32))
        assert all(ctx.lib.gh_touched_lately(ctx.h, p) for p in at)
        for p in at:
            ctx.free(p)


def test_replayed(ctx):
    batch, n_in, n_out = 128, 1152, 625
    rng = np.random.default_rng(6)
    x, dy, w = (rng.standard_normal(s).astype(np.float32) for s in ((batch, n_in), (batch, n_out), (n_in, n_out)))
    at = [ctx.upload(a) for a in (x, dy, w)]
    dw, dx = ctx.upload(np.zeros_like(w)), ctx.upload(np.zeros_like(x))
    cmds = _commands(*at, dw, dx, batch, n_in, n_out, _ffi.F32)
    ctx.run(cmds)
    want = [ctx.d2h(dw, w.shape), ctx.d2h(dx, x.shape)]
    ctx.graph_begin()
    ctx.submit(cmds)
    graph = ctx.graph_end()
    for _ in range(3):
        ctx.h2d(dw, np.zeros_like(w))
        ctx.h2d(dx, np.zeros_like(x))
        ctx.graph_launch(graph)
        ctx.sync()
        for a, b in zip([ctx.d2h(dw, w.shape), ctx.d2h(dx, x.shape)], want):
            assert_bits_equal(a, b)
    ctx.graph_destroy(graph)
    for p in at + [dw, dx]:
        ctx.free(p)
