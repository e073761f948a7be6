"""Small inputs that a run reads where the host wrote them: what an operator makes of one in its own register lies in
device memory, whatever overwrites whatever, and every run gives the numbers of the run that copies."""
import numpy as np
import pytest

from gorgonia_amd import graph as G
from gorgonia_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.fixture()
def engine():
    e = Engine()
    e.Init(0, 1 << 20)
    probe = e.Get(64)
    e.arena = (probe, probe + (5 << 19))   # 2.5 times what was asked for
    e.Put(probe, 64)
    yield e
    e.Close()
    e.destroy()


def _graph(build, shape, np_dt):
    rng = np.random.default_rng(shape[-1])
    g = G.NewGraph()
    x = G.NewTensor(g, np.zeros(shape, np_dt))
    w = G.NewTensor(g, rng.standard_normal(shape).astype(np_dt), resident=True)
    first, last = build(x, w)
    return g, x, first, G.Read(last)


def _scalar(x, value):
    return G.NewScalar(x.g, value, dtype=x.dtype)


def _overwrite(x, w):   # the product takes x's register, the softmax reads it there
    p = G.HadamardProd(x, w)
    return p, G.SoftMax(p)


def _overwrite_twice(x, w):
    p = G.Tanh(G.HadamardProd(x, w))
    return p, G.SoftMax(p)


def _twice_the_same(x, w):
    p = G.HadamardProd(x, x)
    return p, G.SoftMax(G.Add(p, w))


def _by_scalar(x, w):
    p = G.HadamardProd(_scalar(x, 0.5), x)
    return p, G.SoftMax(G.Add(p, w))


def _gradient(x, w):    # masked in place: the second operand's register
    p = G.RectifyDiff(w, x)
    return p, G.SoftMax(p)


@pytest.mark.parametrize("np_dt", [np.float32, np.float64])
@pytest.mark.parametrize("build", [_overwrite, _overwrite_twice, _twice_the_same, _by_scalar, _gradient])
@pytest.mark.parametrize("shape", [(1, 5), (7, 33), (2, 500)])
def test_results_in_an_inputs_register_are_on_the_device(engine, build, shape, np_dt):
    rng = np.random.default_rng(1)
    values = [rng.standard_normal(shape).astype(np_dt) for _ in range(5)]
    want = []
    for v in values:   # the input resident: nothing is read over the bus
        g = G.NewGraph()
        x = G.NewTensor(g, v, resident=True)
        w = G.NewTensor(g, np.random.default_rng(shape[-1]).standard_normal(shape).astype(np_dt), resident=True)
        out = G.Read(build(x, w)[1])
        m = G.NewTapeMachine(g)
        m.RunAll()
        want.append(out.copy())
        m.Close()
    for kw in ({}, {"graph_replay": True}, {"fuse_activations": True}):
        g, x, first, out = _graph(build, shape, np_dt)
        m = G.NewTapeMachine(g, engine=engine, **kw)
        for v, ref in zip(values, want):
            G.Let(x, v)
            m.RunAll()
            assert np.array_equal(out, ref), kw
            assert engine.arena[0] <= m.register_address(first) < engine.arena[1], kw
        m.Close()
