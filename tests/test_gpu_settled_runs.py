"""A tape machine whose runs have settled submits the commands it recorded instead of walking its program: every
run still has to bring the value bound last, see what happened to the arena, and give the numbers of a first run."""
import numpy as np
import pytest

from gorgonia_amd import graph as G
from gorgonia_amd.engine import Engine

pytestmark = pytest.mark.gpu


def _mlp(rows, cols, np_dt, **kw):
    rng = np.random.default_rng(rows)
    g = G.NewGraph()
    x = G.NewTensor(g, np.zeros((rows, cols), np_dt))
    w = G.NewTensor(g, rng.standard_normal((cols, 7)).astype(np_dt), resident=True)
    b = G.NewTensor(g, rng.standard_normal((1, 7)).astype(np_dt), resident=True)
    h = G.BroadcastAdd(G.Mul(x, w), b) if rows > 1 else G.Add(G.Mul(x, w), b)
    out = G.Read(G.Tanh(G.Rectify(h)))
    return g, x, out, G.NewTapeMachine(g, fuse_activations=True, **kw)


def _values(rows, cols, np_dt, n=7):
    rng = np.random.default_rng(5)
    return [rng.standard_normal((rows, cols)).astype(np_dt) for _ in range(n)]


# inputs read in place (to 8 KiB), copied by a command, uploaded in pieces
@pytest.mark.parametrize("np_dt", [np.float32, np.float64])
@pytest.mark.parametrize("rows,cols", [(1, 33), (2, 1024), (1, 2049), (3, 1024), (1024, 1031)])
@pytest.mark.parametrize("replay", [False, True, "measured"])
def test_every_run_takes_the_value_bound_last(rows, cols, np_dt, replay):
    values = _values(rows, cols, np_dt)
    want = []
    for v in values:
        g, x, out, m = _mlp(rows, cols, np_dt)
        G.Let(x, v)
        m.RunAll()
        want.append(out.copy())
        m.Close()
    g, x, out, m = _mlp(rows, cols, np_dt, graph_replay=replay)
    for v, w in zip(values, want):
        G.Let(x, v)
        m.RunAll()
        assert np.array_equal(out, w)
    m.Close()


def test_arena_used_between_runs_and_lending_switched():
    values = _values(4, 300, np.float32)
    g, x, out, m = _mlp(4, 300, np.float32)
    e, held = m.engine(), []
    for i, v in enumerate(values * 2):
        G.Let(x, v)
        m.RunAll()
        first = out.copy()
        if i % 3 == 0:
            held.append(e.to_device(np.full(64, i, np.float32)))   # a hole of the arena the next run would have used
        elif i % 3 == 1:
            G.LetBorrowed(x)
            m.input(x)[...] = v
            m.RunAll()
            assert np.array_equal(out, first) and np.array_equal(m.input(x), v)
        assert all(np.array_equal(e.to_host(t), np.full(64, 3 * k, np.float32)) for k, t in enumerate(held))
        ref = _mlp(4, 300, np.float32)
        G.Let(ref[1], v)
        ref[3].RunAll()
        assert np.array_equal(first, ref[2])
        ref[3].Close()
    m.Close()


def test_two_settled_machines_on_one_engine():
    e = Engine()
    e.Init(0, 1 << 20)
    values = _values(2, 64, np.float32)
    one, two = _mlp(2, 64, np.float32, engine=e), _mlp(2, 64, np.float32, engine=e)
    for v in values:
        for g, x, out, m in (one, two, two):
            G.Let(x, v)
            m.RunAll()
        assert np.array_equal(one[2], two[2])
        m = _mlp(2, 64, np.float32)
        G.Let(m[1], v)
        m[3].RunAll()
        assert np.array_equal(one[2], m[2])
        m[3].Close()
    for g, x, out, m in (one, two):
        m.Close()
    e.Close()
    e.destroy()
