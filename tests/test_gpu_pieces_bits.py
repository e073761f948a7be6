"""A batch in pieces (gh_pieces.hip) has the bits of the batch uploaded whole: as commands, and on a tape machine in every replay
mode."""
import ctypes as C

import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from gorgonia_amd import graph as G
from tests.test_gpu_pieces import _Host
from tests.util import assert_bits_equal

pytestmark = pytest.mark.gpu


class _Chain:
    """Convolutions with batch normalisation, an activation and a 2x2 pooling, in the epilogue where the library offers that."""

    def __init__(self, ctx, B, H, W, channels, act="leaky"):
        self.ctx, self.B, self.mem, self.results = ctx, B, [], []
        r = np.random.default_rng(B + H + W)
        self.shape = (B, channels[0], H, W)
        self.nbytes = 4 * int(np.prod(self.shape))
        self.x = at = self._new(np.zeros(self.shape, np.float32))
        self.layers = []
        h, w = H, W
        for c, f in zip(channels, channels[1:]):
            filters = self._new(r.standard_normal((f, c, 3, 3)).astype(np.float32) / np.float32(np.sqrt(9 * c)))
            bn = [self._new(v.astype(np.float32)) for v in (r.standard_normal(f), r.uniform(0.5, 2, f), r.standard_normal(f), r.standard_normal(f))]
            y = self._result(B, f, h, w)
            z = self._result(B, f, h // 2, w // 2)
            kw = dict(act=act, alpha=0.1, bn=bn)
            pooled = D.cmd_conv2d(at, filters, z, B, c, h, w, f, 3, 3, (1, 1), pool2=True, **kw)
            if ctx.lib.gh_conv2d_can_pool(C.byref(pooled)):
                self.layers.append(pooled)
            else:
                self.layers += [D.cmd_conv2d(at, filters, y, B, c, h, w, f, 3, 3, (1, 1), **kw), D.cmd_maxpool2d(y, z, B, f, h, w, 2, 2, (0, 0), (2, 2))]
            at, h, w = z, h // 2, w // 2

    def _new(self, v):
        self.mem.append(self.ctx.upload(v))
        return self.mem[-1]

    def _result(self, *shape):
        self.results.append((self._new(np.full(shape, np.nan, np.float32)), shape))
        return self.results[-1][0]

    def run(self, host):
        for p, shape in self.results:
            self.ctx.h2d(p, np.full(shape, np.nan, np.float32))
        cmds = [D.cmd_copy(self.x, host.value, self.nbytes)] + self.layers
        self.ctx.submit(cmds)
        self.ctx.sync()
        return [self.ctx.d2h(p, shape) for p, shape in self.results], self.ctx.lib.gh_pieces_layers((_ffi.GhCmd * len(cmds))(*cmds), len(cmds))

    def close(self):
        for p in self.mem:
            self.ctx.free(p)


# B, H, W, channels, and the layers that run in pieces: a detector's (the last in pieces on k_conv3x3_patch, on k_conv3x3_lanes had
# the piece its own choice), batches that the pieces do not divide, odd extents, layers for k_conv3x3_lanes in each of its orders
DETECTOR = (3, 16, 32, 64, 128)
CASES = [(8, 416, 416, DETECTOR, 5), (7, 384, 384, DETECTOR, 4), (5, 384, 384, DETECTOR, 4), (3, 416, 416, DETECTOR, 3), (2, 416, 416, DETECTOR, 3), (8, 320, 320, DETECTOR, 4),
         (7, 331, 333, DETECTOR, None), (32, 112, 110, (4, 8, 64, 96, 128), None), (8, 130, 130, (16, 32, 32, 64), None), (9, 52, 52, (64, 128, 64), None),
         (3, 104, 104, (32, 64, 128), None), (40, 26, 26, (64, 64, 128), None)]


@pytest.mark.parametrize("B,H,W,channels,layers", CASES)
def test_commands(ctx, monkeypatch, B, H, W, channels, layers):
    chain = _Chain(ctx, B, H, W, channels)
    x = np.random.default_rng(1).uniform(0, 1, chain.shape).astype(np.float32)
    x[B - 1] = x[0]   # an image of the first piece and one of the last
    host = _Host(ctx, chain.nbytes)
    host.fill(x)
    before = ctx.joint_launches(_ffi.JOINT_PIECES)[0]
    got, answer = chain.run(host.p)
    launches, form = ctx.joint_launches(_ffi.JOINT_PIECES)
    if layers is not None:
        assert answer == layers
    assert launches - before == (answer > 0) and (not answer or form % 100 == answer)
    monkeypatch.setenv("GORGONIA_HIP_NO_PIECES", "1")
    want, _ = chain.run(host.p)
    assert ctx.joint_launches(_ffi.JOINT_PIECES)[0] == launches
    for g, w in zip(got, want):
        assert_bits_equal(g, w)
        assert_bits_equal(g[B - 1], g[0])
    host.close()
    chain.close()


@pytest.mark.parametrize("mode", [False, True, "measured"])
def test_tape(monkeypatch, mode):
    """A lent batch of several megabytes: the same bits in each of a machine's runs, eager, captured and replayed."""
    B, S = 8, 416
    r = np.random.default_rng(3)
    x = r.uniform(0, 1, (B, 3, S, S)).astype(np.float32)
    ws = [r.standard_normal((f, c, 3, 3)).astype(np.float32) / np.float32(np.sqrt(9 * c)) for c, f in zip(DETECTOR, DETECTOR[1:])]

    def machine(graph_replay):
        g = G.NewGraph()
        node = h = G.LetBorrowed(G.NewTensor(g, x))
        for w in ws:
            h = G.MaxPool2D(G.LeakyRelu(G.Conv2d(h, G.NewTensor(g, w, resident=True), (3, 3), (1, 1), (1, 1), (1, 1)), 0.1), (2, 2), (0, 0), (2, 2))
        for _ in range(3):   # enough commands for a graph
            h = G.Rectify(G.Add(h, h))
        out = G.Read(h)
        m = G.NewTapeMachine(g, graph_replay=graph_replay, fuse_activations=True)
        m.input(node)[...] = x
        return m, out
    with monkeypatch.context() as p:
        p.setenv("GORGONIA_HIP_NO_PIECES", "1")
        m, out = machine(False)
        m.RunAll()
        want = out.copy()
        m.Close()
    m, out = machine(mode)
    for run in range(8):
        out[...] = np.nan
        m.RunAll()
        assert_bits_equal(out, want, (mode, run))
    launches, form = m.engine().joint_launches(_ffi.JOINT_PIECES)
    assert form % 100 >= 4 and (launches == 7 if not mode else launches >= 1)   # (the first run uploads the filters as well)
    m.Close()


def test_tape_with_filters_that_are_not_resident(monkeypatch):
    """Filters uploaded in front of a lent batch by each run: their memory is not given to a result that a first piece writes while
    the next one still reads them."""
    B, S = 16, 52
    r = np.random.default_rng(4)
    x = r.uniform(-1, 1, (B, 64, S, S)).astype(np.float32)
    ws = [r.standard_normal(s).astype(np.float32) / 24 for s in ((128, 64, 3, 3), (64, 128, 3, 3))]

    def run():
        g = G.NewGraph()
        w = [G.NewTensor(g, v) for v in ws]
        node = G.LetBorrowed(G.NewTensor(g, x))
        h = G.MaxPool2D(G.Conv2d(node, w[0], (3, 3), (1, 1), (1, 1), (1, 1)), (2, 2), (0, 0), (2, 2))
        out = G.Read(G.Rectify(G.Conv2d(h, w[1], (3, 3), (1, 1), (1, 1), (1, 1))))
        m = G.NewTapeMachine(g)
        m.input(node)[...] = x
        got = []
        for k in range(3):
            G.Let(w[0], ws[0] * np.float32(k + 1))
            m.RunAll()
            got.append(out.copy())
        form = m.engine().joint_launches(_ffi.JOINT_PIECES)
        m.Close()
        return got, form
    got, (launches, form) = run()
    monkeypatch.setenv("GORGONIA_HIP_NO_PIECES", "1")
    want, none = run()
    assert none[0] == 0 and launches == 3 and form % 100 == 3, (launches, form)
    for g, w in zip(got, want):
        assert_bits_equal(g, w)
