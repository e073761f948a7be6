"""Which small inputs a tape machine leaves in pinned memory: those that are read once, wherever that is and however
often, and not those that a kernel walks along, passes over repeatedly or writes."""
import numpy as np
import pytest

from gorgonia_amd import graph as G


def _in_place(x, out, **kw):
    G.Read(out)
    m = G.NewTapeMachine(x.g, compile_only=True, **kw)
    lines = [l for l in m.program().splitlines() if "devTrans node %d " % x.id in l]
    m.Close()
    assert len(lines) == 1
    return "[in place]" in lines[0]


def _input(g, *shape, dtype=np.float32, **kw):
    return G.NewTensor(g, np.ones(shape, dtype), **kw)


def test_elementwise_readers():
    for rows in (2, 512):   # however many workgroups read it
        g = G.NewGraph()
        big, row = _input(g, rows, 2048, resident=True), _input(g, 1, 2048)
        assert _in_place(row, G.Tanh(G.BroadcastAdd(big, row)))
    g = G.NewGraph()
    x = _input(g, 16, 128)
    assert _in_place(x, G.SoftMax(G.HadamardProd(x, _input(g, 16, 128, resident=True))))
    g = G.NewGraph()
    x = _input(g, 17, 128)   # 8704 bytes
    assert not _in_place(x, G.Tanh(x))
    g = G.NewGraph()
    x = _input(g, 16, 128)
    assert not _in_place(x, G.SoftMax(x))   # several passes
    g = G.NewGraph()
    x = _input(g, 16, 128, resident=True)
    assert not _in_place(x, G.Tanh(x))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_products(dtype):
    line = 2048 // np.dtype(dtype).itemsize   # values along K
    for k in (line, line + 1):
        g = G.NewGraph()
        a = _input(g, 1, k, dtype=dtype)
        assert _in_place(a, G.Mul(a, _input(g, k, 40, dtype=dtype, resident=True))) == (k <= line)
        g = G.NewGraph()
        b = _input(g, k, 1, dtype=dtype)
        assert _in_place(b, G.Mul(_input(g, 50, k, dtype=dtype, resident=True), b)) == (k <= line)
        g = G.NewGraph()
        a = _input(g, k, 1, dtype=dtype)   # transposed: K is the first axis
        assert _in_place(a, G.Mul(a, _input(g, k, 40, dtype=dtype, resident=True), transA=True)) == (k <= line)
        g = G.NewGraph()
        v = _input(g, k, dtype=dtype)
        assert _in_place(v, G.Mul(_input(g, 50, k, dtype=dtype, resident=True), v)) == (k <= line)
    g = G.NewGraph()
    a = _input(g, 1, 1024, dtype=dtype)   # many columns hide the walk
    assert _in_place(a, G.Mul(a, _input(g, 1024, 2049, dtype=dtype, resident=True)))
    # one reader that walks along it is enough, through a view as well
    g = G.NewGraph()
    x = _input(g, 3, 600)
    view = G.Reshape(x, (1, 1800))
    G.Read(G.Mul(view, _input(g, 1800, 5, resident=True)))
    assert not _in_place(x, G.Tanh(x))


def test_convolutions_and_folded_operands():
    for c, hw, kept in ((1, 22, True), (1, 23, False), (2, 30, True)):
        g = G.NewGraph()
        x = _input(g, 1, c, hw, hw)
        assert _in_place(x, G.Conv2d(x, _input(g, 8, c, 3, 3, resident=True), (3, 3), (1, 1), (1, 1), (1, 1))) == kept
    g = G.NewGraph()
    w = _input(g, 16, 3, 3, 3)
    assert _in_place(w, G.Rectify(G.Conv2d(_input(g, 2, 3, 40, 40, resident=True), w, (3, 3), (1, 1), (1, 1), (1, 1))), fuse_activations=True)
    g = G.NewGraph()
    bias = _input(g, 1, 700)
    x, w = _input(g, 30, 800, resident=True), _input(g, 800, 700, resident=True)
    assert _in_place(bias, G.BroadcastAdd(G.Mul(x, w), bias), fuse_activations=True)


def test_what_is_written_is_not_left_there():
    g = G.NewGraph()
    w, grad = _input(g, 8, 8), _input(g, 8, 8, resident=True)
    corrections = G.NewTensor(g, G.AdamCorrections(1))
    caches = [_input(g, 8, 8) for _ in range(2)]
    step = G.SolverStep("adam", w, grad, caches, corrections=corrections)
    G.Read(step)
    m = G.NewTapeMachine(g, compile_only=True)
    prog = [l for l in m.program().splitlines() if "[in place]" in l]
    m.Close()
    assert len(prog) == 1 and "node %d " % corrections.id in prog[0]
    g = G.NewGraph()
    x, v = _input(g, 4, 4), _input(g, 4, 4, resident=True)
    G.Set(x, v)
    assert not _in_place(x, G.Tanh(x))
