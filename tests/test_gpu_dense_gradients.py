"""A dense layer's weight gradient and input gradient in one launch (k_gemm_gradients.hip): the bits of the two products
submitted apart, in both orders, and of what lies around their results."""
import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.util import assert_bits_equal

pytestmark = pytest.mark.gpu

# (batch, inputs, outputs) and the kernel that runs both (gh_joint_launches), None where each has a launch: every pair of kernels that a
# draw of 13000 found, tiles that the sizes fill and do not, the smallest contractions, and products that one launch has no kernel for
F32 = {
    (128, 1152, 625): 1401020162, (128, 625, 10): 2008114010, (8, 1152, 625): 1401010080, (8, 625, 10): None, (31, 1152, 625): 1401020161,
    (33, 625, 10): 2008114010, (49, 1152, 625): 1401020162, (200, 1152, 625): None, (64, 784, 300): 2008220081, (64, 300, 100): 2008120081,
    (64, 100, 10): 2008114010, (37, 99, 41): 2008120081, (17, 530, 513): 1401020161, (16, 33, 600): 1401020161, (100, 47, 515): 2008120161,
    (5, 7, 9): 1401014010, (4, 16, 4): 1401014010, (300, 1152, 625): None, (2, 700, 10): None, (90, 2000, 30): 2008114010,
    (15, 400, 300): 1401010080, (9, 37, 333): 1401010080, (12, 2500, 140): 1401010080, (84, 751, 705): 1401020162, (66, 2860, 326): 1501010080,
    (29, 5192, 229): 1501020082, (29, 999, 1092): 1501020161, (46, 2049, 558): 1501020162, (25, 204, 33): 1401020081, (17, 2615, 33): 1401020082,
    (35, 24, 920): 2008120161, (87, 741, 32): 2008120082, (168, 1414, 35): 2008214010, (45, 1048, 50): 2008220081, (34, 1722, 38): 2008220082,
    (43, 216, 763): 2008220161, (271, 231, 848): 2008220162, (49, 31, 1): 2008114010}
F64 = {
    (50, 1152, 625): 1200020081, (50, 625, 10): 1000010000, (8, 1152, 625): None, (96, 1152, 625): 1200020081, (96, 625, 10): 2004110000,
    (13, 777, 300): 1000020081, (64, 300, 100): 2004120041, (100, 515, 77): 2004120041, (3, 5, 2): 1000010000, (70, 65, 260): 2004120081,
    (129, 31, 64): 2004120041, (64, 500, 3000): 1100020081, (40, 1600, 1600): None, (24, 2000, 2000): None, (2, 64, 3): 1000010000,
    (51, 778, 2019): 1000020081, (2, 4362, 33): 1100010000, (2, 1464, 177): 1100020041, (97, 1954, 713): 1200010000, (3, 2049, 246): 1200020041,
    (163, 1289, 594): 1300010000, (39, 5223, 141): 1300020041, (106, 1764, 1371): 1400010000, (33, 1158, 1024): 1400020081, (67, 7, 3): 2004110000,
    (2, 362, 80): 1000020041, (37, 877, 931): 1300020081,
    # weight gradients in eight slices
    (682, 296, 610): 1008010000, (1448, 96, 1582): 1008020081, (708, 335, 1002): 1108010000, (641, 480, 675): 1108020081,
    (1578, 133, 3666): 1208010000, (655, 186, 2987): 1208020081, (665, 345, 2324): 1308010000, (730, 251, 3435): 1308020081,
    (723, 312, 3489): 1408010000, (944, 277, 3673): 1408020081}
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
            before = ctx.joint_launches(_ffi.JOINT_DENSE_GRADIENTS)[0]
            ctx.run(cmds)
            after, form = ctx.joint_launches(_ffi.JOINT_DENSE_GRADIENTS)
            want = (F32 if dt == np.float32 else F64)[batch, n_in, n_out]
            assert after - before == (want is not None) and want in (None, form)
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


def test_tuning_switch(ctx, monkeypatch):
    """GORGONIA_HIP_GEMM_APART: a launch each."""
    monkeypatch.setenv("GORGONIA_HIP_GEMM_APART", "1")
    at = [ctx.upload(np.ones(1250, np.float32)) for _ in range(5)]
    before = ctx.joint_launches(_ffi.JOINT_DENSE_GRADIENTS)
    ctx.run(_commands(*at, 64, 15, 10, _ffi.F32))
    assert ctx.joint_launches(_ffi.JOINT_DENSE_GRADIENTS) == before
    monkeypatch.delenv("GORGONIA_HIP_GEMM_APART")
    ctx.run(_commands(*at, 64, 15, 10, _ffi.F32))
    assert ctx.joint_launches(_ffi.JOINT_DENSE_GRADIENTS)[0] == before[0] + 1
    for p in at:
        ctx.free(p)


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
