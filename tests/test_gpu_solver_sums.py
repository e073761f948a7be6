"""Solver steps that take the waiting sums of their gradients along (k_solver.hip): the bits of one submission for each command,
also where a sum has to do with the steps in another way."""
import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.test_gpu_slab_sums import LAYERS, _gradient, _same, _Tensors

pytestmark = pytest.mark.gpu

SETTINGS = {"vanilla": (0.01, 0.0, 1e-3, 1e-4, 0.5, 0.25, 0.0, 0.0, 0.0, 0.0), "rmsprop": (1e-3, 1e-8, 0.0, 1e-6, 5.0, 0.0, 0.999, 0.001, 0.0, 0.0),
            "adam": (1e-3, 1e-8, 1e-3, 1e-4, 0.0, 0.0, 0.9, 0.999, 1.2, 1.1)}
USE = {"vanilla": 15, "rmsprop": 6, "adam": 3}
TYPES = [(_ffi.F32, np.float32), (_ffi.F64, np.float64)]


def _step(t, kind, w, g, n, code=_ffi.F32):
    return D.cmd_solver_step(kind, w, g, n, SETTINGS[kind], USE[kind], cache=_positive(t, n), cache2=_positive(t, n), dtype=code)


def _positive(t, n):
    p = t.ctx.upload(np.abs(t.rng.standard_normal(n)).astype(t.dt))
    t.all.append((p, (n,)))
    return p


def _size(layer):
    return layer[4] * layer[1] * 9


@pytest.mark.parametrize("kind", SETTINGS)
@pytest.mark.parametrize("code,np_dt", TYPES)
def test_steps_behind_their_gradients(ctx, kind, code, np_dt):
    """Sums of every kind, a tensor whose gradient is none, and a copy behind the steps."""
    def build(t):
        grads = [_gradient(t, layer, code) for layer in LAYERS]
        steps = [_step(t, kind, t.make(_size(layer)), g.ptr[2], _size(layer), code) for g, layer in zip(grads[1:], LAYERS[1:])]
        steps.insert(3, _step(t, kind, t.make(777), t.make(777), 777, code))
        return grads + steps + [D.cmd_copy(t.make(300), t.make(300), 300 * np_dt().itemsize)]
    before = ctx.joint_launches(_ffi.JOINT_SOLVER_SUMS)[0]
    _same(ctx, build, np_dt)
    # six of the seven gradients that have a step waited for it
    assert ctx.joint_launches(_ffi.JOINT_SOLVER_SUMS) == (before + 1, 6)


@pytest.mark.parametrize("form", ["one", "two for one", "part", "weights", "cache", "copy", "other type", "three, two stepped"])
def test_other_forms(ctx, form):
    layer = (8, 16, 52, 52, 32)
    n = _size(layer)

    def build(t):
        g = _gradient(t, layer)
        dw = g.ptr[2]
        if form == "one":
            return [g, _step(t, "rmsprop", t.make(n), dw, n)]
        if form == "two for one":
            return [g, _step(t, "adam", t.make(n), dw, n), _step(t, "adam", t.make(n), dw, n)]
        if form == "part":
            return [g, _step(t, "vanilla", t.make(n), dw, n - 5), _step(t, "vanilla", t.make(9), t.make(9), 9)]
        if form == "weights":   # the gradient is what the second step changes
            return [g, _step(t, "vanilla", dw, t.make(n), n)]
        if form == "cache":
            s = _step(t, "rmsprop", t.make(n), t.make(n), n)
            s.ptr[2] = dw
            return [g, s]
        if form == "copy":
            return [g, _step(t, "vanilla", t.make(n), dw, n), D.cmd_copy(t.make(100), dw + 64, 400)]
        if form == "other type":
            w, g64 = t.make(2 * n), t.make(2 * n)
            return [g, _step(t, "vanilla", t.make(n), dw, n), _step(t, "vanilla", w, g64, n, _ffi.F64)]
        second, third = _gradient(t, (64, 32, 14, 14, 64)), _gradient(t, (8, 64, 26, 26, 128))
        return [g, second, third, _step(t, "adam", t.make(n), dw, n), _step(t, "adam", t.make(64 * 32 * 9), second.ptr[2], 64 * 32 * 9)]
    before = ctx.joint_launches(_ffi.JOINT_SOLVER_SUMS)[0]
    _same(ctx, build)
    after, steps = ctx.joint_launches(_ffi.JOINT_SOLVER_SUMS)
    want = {"one": 1, "other type": 1, "three, two stepped": 2}.get(form)   # steps that took their sum along
    assert after - before == (want is not None) and want in (None, steps)


@pytest.mark.parametrize("kind", SETTINGS)
@pytest.mark.parametrize("form", ["gradient from weights", "weights from gradient", "same cache", "overlap", "the same weights"])
def test_steps_that_have_to_do_with_each_other(ctx, kind, form):
    """The second of two steps reads or writes what the first writes, or writes what it reads: in the order of the commands."""
    n = 300000

    def build(t):
        first, free = _step(t, kind, t.make(n + 64), t.make(n), n), _step(t, kind, t.make(n), t.make(n), n)
        w, g = {"gradient from weights": (t.make(n), first.ptr[0]), "weights from gradient": (first.ptr[1], t.make(n)), "same cache": (t.make(n), t.make(n)),
                "overlap": (first.ptr[0] + 256, t.make(n)), "the same weights": (first.ptr[0], t.make(n))}[form]
        second = _step(t, kind, w, g, n)
        if form == "same cache":
            second.ptr[2] = first.ptr[2]
        return [first, free, second]
    _same(ctx, build)


def test_operands_of_one_step_are_in_the_cache_account():
    layer = (8, 16, 52, 52, 32)
    n = _size(layer)
    with D.Context() as ctx:
        t = _Tensors(ctx, np.float32)
        gradient = _gradient(t, layer)
        step = _step(t, "adam", t.make(n), gradient.ptr[2], n)
        assert not any(ctx.lib.gh_touched_lately(ctx.h, p) for p, _ in t.all)
        ctx.run([gradient, step])
        assert all(ctx.lib.gh_touched_lately(ctx.h, p) for p, _ in t.all)
        t.values()


def test_replayed(ctx):
    layer = (8, 16, 52, 52, 32)
    n = _size(layer)
    rng = np.random.default_rng(3)
    x, dy, w = (rng.standard_normal(s).astype(np.float32) for s in ((8, 16, 52, 52), (8, 32, 52, 52), n))
    got = []
    for replay in (False, True):
        at = [ctx.upload(a) for a in (x, dy, w, np.zeros(n, np.float32), np.zeros(n, np.float32))]
        cmds = [D.cmd_conv2d_bwd_filter(at[0], at[1], at[3], 8, 16, 52, 52, 32, 3, 3, pad=(1, 1)),
                D.cmd_solver_step("rmsprop", at[2], at[3], n, SETTINGS["rmsprop"], USE["rmsprop"], cache=at[4])]
        ctx.run(cmds)
        if replay:
            ctx.graph_begin()
            ctx.submit(cmds)
            graph = ctx.graph_end()
        values = []
        for _ in range(3):
            if replay:
                ctx.graph_launch(graph)
                ctx.sync()
            else:
                ctx.run(cmds)
            values += [ctx.d2h(at[i], (n,)) for i in (2, 3, 4)]
        if replay:
            ctx.graph_destroy(graph)
        got.append(values)
        for p in at:
            ctx.free(p)
    for a, b in zip(*got):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
