"""Batch statistics with the pooling behind them and their gradients in one launch (k_bn_held.hip): every tensor that the two
commands write.  The forward's are those of the two commands apart, to the bit; the saved statistics are held to a float64 sum,
what is computed from them to the bit; the gradient's two sums are not stored, so that its result is held to the bound that
their rounding leaves."""
import threading
import time

import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.util import assert_bits_equal, rel_frobenius

pytestmark = pytest.mark.gpu

EPS, MOMENTUM = 1e-5, 0.1
# a value passes at most 72 additions in its thread (of the shapes below), 6 in its wavefront, 3 and 64 behind it
DEPTH = 150
U = 2.0 ** -24
# four columns a load with one to three units a thread, two columns with one to six, single loads (an odd size), one workgroup a
# channel and sixty-four, a window for each channel, more channels than half of the compute units
SHAPES = [(2, 3, 4, 4), (8, 16, 104, 104), (8, 16, 160, 160), (8, 16, 208, 208), (8, 128, 26, 26), (8, 16, 102, 102), (8, 16, 202, 202), (8, 128, 25, 25),
          (3, 16, 207, 207), (4, 2, 64, 64), (8, 4, 256, 256), (1, 4, 300, 300), (2, 5, 2, 2), (1, 1, 3, 2), (3, 250, 9, 8), (2, 256, 6, 6), (1, 128, 2, 3)]


class _Place:
    """One allocation with named tensors, each `shift` elements from a 16-byte boundary."""

    def __init__(self, ctx, shift, **arrays):
        self.ctx, self.at, self.shape, n, flat = ctx, {}, {}, 0, []
        for k, a in arrays.items():
            pre = np.full(4 + shift, np.nan, np.float32)
            flat += [pre, a.ravel(), np.full(-(a.size + shift) % 4, np.nan, np.float32)]
            self.at[k], self.shape[k] = n + pre.size, a.shape
            n += pre.size + a.size + flat[-1].size
        self.n, self.base = n, ctx.upload(np.concatenate(flat))

    def __getitem__(self, k):
        return self.base + 4 * self.at[k]

    def all(self):
        whole = self.ctx.d2h(self.base, (self.n,), np.float32)
        self.ctx.free(self.base)
        return {k: whole[a:a + int(np.prod(self.shape[k]))].reshape(self.shape[k]) for k, a in self.at.items()}


def _inputs(shape, seed):
    r = np.random.default_rng(seed)
    B, C, H, W = shape
    x = (np.round(r.standard_normal(shape) * 8) / 8 + r.uniform(-1, 1, (1, C, 1, 1))).astype(np.float32)   # ties in windows
    chan = lambda: r.uniform(0.5, 1.5, C).astype(np.float32)
    return x, chan(), chan(), r.standard_normal((B, C, H // 2, W // 2)).astype(np.float32)


def _relu(v):
    return v * (v >= 0).astype(np.float32)


def _windows(v):
    H, W = v.shape[2] // 2 * 2, v.shape[3] // 2 * 2
    return np.stack([v[:, :, a:H:2, b:W:2] for a in (0, 1) for b in (0, 1)])


def _commands(m, shape, z="x", dz="dz"):
    B, C, H, W = shape
    bn = D.cmd_bn_train(m["x"], m["y"], m["rm"], m["rv"], m["sm"], m["sv"], B, C, H * W, EPS, MOMENTUM)
    pool = D.cmd_maxpool2d(m["y"], m["p"], B, C, H, W, 2, 2, (0, 0), (2, 2))
    back = D.cmd_maxpool2d_bwd(m["y"], m["dp"], m["t"], B, C, H, W, 2, 2, (0, 0), (2, 2))
    pool.flags |= _ffi.FLAG_ACT_RELU
    back.flags |= _ffi.FLAG_ACT_RELU
    return [bn, pool], [back, D.cmd_bn_bwd(m[z], m["t"], m[dz], m["sm"], m["sv"], B, C, H * W, EPS)]


def _run(ctx, shape, seed, shift=0, dz="dz", polls=None, monkeypatch=None, together=True, forward=True):
    x, rm, rv, dp = _inputs(shape, seed)
    nan = np.full_like(x, np.nan)
    m = _Place(ctx, shift, x=x, y=nan, p=np.full_like(dp, np.nan), rm=rm, rv=rv, sm=np.full_like(rm, np.nan), sv=np.full_like(rm, np.nan), dp=dp, t=nan, dz=nan)
    if polls is not None:
        monkeypatch.setenv("GORGONIA_HIP_BN_POLLS", str(polls))
    fwd, bwd = _commands(m, shape, dz=dz)
    for group in ([fwd] if forward else [[c] for c in fwd]):
        ctx.run(group)
    for group in ([bwd] if together else [[c] for c in bwd]):
        ctx.run(group)
    return (x, rm, rv, dp), m.all()


def _check(shape, given, got, dz="dz"):
    (x, rm, rv, dp), (B, C, H, W) = given, shape
    n = np.float32(B * H * W)
    f32 = np.float32
    x64 = x.astype(np.float64)
    mean64 = x64.mean((0, 2, 3))
    # the mean's rounding, and what is left of it in the sum of squares (n d^2), besides that sum's own
    d = DEPTH * U * np.abs(x64).mean((0, 2, 3))
    assert np.all(np.abs(got["sm"] - mean64) <= d + U * np.abs(mean64))
    dev = x64 - got["sm"].astype(np.float64)[None, :, None, None]
    var64 = (dev ** 2).sum((0, 2, 3))
    assert np.all(np.abs(got["sv"] - var64) <= (DEPTH + 4) * U * var64)
    sm, sv = got["sm"], got["sv"]
    with np.errstate(divide="ignore", invalid="ignore"):
        assert_bits_equal(got["rm"], f32(MOMENTUM) * sm + (f32(1) - f32(MOMENTUM)) * rm)
        assert_bits_equal(got["rv"], f32(MOMENTUM) * (sv / f32(B * H * W - 1)) + (f32(1) - f32(MOMENTUM)) * rv)
    a = f32(1) / np.sqrt(sv / n + f32(EPS))
    y = x * a[None, :, None, None] + (-sm * a)[None, :, None, None]
    if dz != "y":
        assert_bits_equal(got["y"], y)
    win = _windows(_relu(y))
    # the first of the largest; MaxPool2DDiff behind Rectify gives it dy where y >= 0
    first = win.argmax(0)
    assert_bits_equal(got["p"], np.take_along_axis(win, first[None], 0)[0])
    t = np.zeros_like(y)
    for k in range(4):
        hit = np.where(first == k, np.float32(0) + dp, np.float32(0))
        t[:, :, k >> 1:H // 2 * 2:2, k & 1:W // 2 * 2:2] = hit * (_windows(y)[k] >= 0)
    assert_bits_equal(got["t"], t)
    g64, invstd = t.astype(np.float64), a.astype(np.float64)[None, :, None, None]
    c = (x64 - sm.astype(np.float64)[None, :, None, None])
    s, dot = g64.sum((0, 2, 3), keepdims=True), (c * g64).sum((0, 2, 3), keepdims=True)
    # x dy - mean dy, each product rounded
    each = np.abs(x64 * g64) + np.abs(sm.astype(np.float64)[None, :, None, None] * g64)
    ds = DEPTH * U * np.abs(g64).sum((0, 2, 3), keepdims=True)
    ddot = (DEPTH + 2) * U * each.sum((0, 2, 3), keepdims=True)
    N = float(n)
    want = (g64 - s / N - c * (dot * invstd ** 2 / N)) * invstd
    size = (np.abs(g64) + np.abs(s) / N + np.abs(c * dot) * invstd ** 2 / N) * invstd
    bound = (ds / N + np.abs(c) * ddot * invstd ** 2 / N) * invstd + 16 * U * (size + invstd * np.abs(x64) * np.abs(dot) * invstd ** 2 / N)
    assert np.all(np.abs(got[dz] - want) <= bound + 1e-38)


@pytest.mark.parametrize("shape", SHAPES)
def test_one_launch(ctx, shape):
    for dz in ("dz", "y"):   # the normalised tensor's gradient in a place of its own, or over the pooled tensor's source
        given, got = _run(ctx, shape, 5, dz=dz)
        _check(shape, given, got, dz)
    _, apart = _run(ctx, shape, 5, forward=False)
    for k in ("y", "p", "sm", "sv", "rm", "rv", "t"):
        if k != "y":   # (the last gradient lies over it)
            assert_bits_equal(got[k], apart[k])


@pytest.mark.parametrize("shape", SHAPES)
def test_gradient_next_to_the_commands_apart(ctx, shape):
    """Two orders of adding the same terms: both within the bound, and apart by less than the rounding of a result."""
    given, got = _run(ctx, shape, 5)
    _, apart = _run(ctx, shape, 5, together=False)
    _check(shape, given, apart)
    for k in ("y", "p", "sm", "sv", "rm", "rv", "t"):
        assert_bits_equal(got[k], apart[k])
    assert rel_frobenius(got["dz"], apart["dz"].astype(np.float64)) <= U


@pytest.mark.parametrize("shift", [1, 2])
def test_single_and_pair_loads(ctx, shift):
    shape = (3, 16, 36, 36)
    given, got = _run(ctx, shape, 6, shift=shift)
    _check(shape, given, got)


@pytest.mark.parametrize("polls", [0, 1])
@pytest.mark.parametrize("shape", [(8, 16, 104, 104), (4, 2, 64, 64), (8, 128, 25, 25), (1, 4, 300, 300)])
def test_a_workgroup_that_does_not_wait(ctx, shape, polls, monkeypatch):
    """The shares that have not come are added up where they are missed, to the bits of those that come."""
    given, got = _run(ctx, shape, 7, polls=polls, monkeypatch=monkeypatch)
    _check(shape, given, got)
    monkeypatch.delenv("GORGONIA_HIP_BN_POLLS")
    _, again = _run(ctx, shape, 7)
    for k in got:
        assert_bits_equal(got[k], again[k])


def test_a_pair_that_overlaps_runs_apart(ctx):
    """dz over the gradient it is computed from: two launches, as before."""
    shape = (4, 16, 32, 32)
    out = [_run(ctx, shape, 8, dz="t", together=together)[1] for together in (True, False)]
    for k in out[0]:
        assert_bits_equal(out[0][k], out[1][k])


def test_replays(ctx):
    """Captured: every replay finds the exchanged sums' places as it needs them."""
    shape = (4, 16, 52, 52)
    x, rm, rv, dp = _inputs(shape, 9)
    nan = np.full_like(x, np.nan)
    m = _Place(ctx, 0, x=x, y=nan, p=np.full_like(dp, np.nan), rm=rm, rv=rv, sm=rm * 0, sv=rm * 0, dp=dp, t=nan, dz=nan)
    fwd, bwd = _commands(m, shape)
    ctx.run(fwd + bwd)
    first = ctx.d2h(m["dz"], x.shape, np.float32)
    ctx.graph_begin()
    ctx.submit(fwd + bwd)
    graph = ctx.graph_end()
    for _ in range(3):
        ctx.h2d(m["dz"], nan)
        ctx.graph_launch(graph)
        ctx.sync()
        assert_bits_equal(ctx.d2h(m["dz"], x.shape, np.float32), first)
        ctx.run(fwd + bwd)
    ctx.graph_destroy(graph)
    m.all()


@pytest.mark.parametrize("shape", [(8, 16, 208, 208), (8, 32, 104, 104)])
def test_time_of_three_contexts_at_once(shape):
    """Each launch has a workgroup for every compute unit: together they find room for some of each.  Three take three times as
    long as one, and some more where they load what another has put out of the caches."""
    x, rm, rv, dp = _inputs(shape, 11)
    nan = np.full_like(x, np.nan)

    def seconds(ctxs):
        work = []
        for c in ctxs:
            m = _Place(c, 0, x=x, y=nan, p=np.full_like(dp, np.nan), rm=rm, rv=rv, sm=rm * 0, sv=rm * 0, dp=dp, t=nan, dz=nan)
            work.append((c, sum(_commands(m, shape), []) * 10))
            c.run(work[-1][1])
        gate = threading.Barrier(len(work) + 1)

        def run(c, cmds):
            gate.wait()
            for _ in range(10):
                c.run(cmds)
            gate.wait()
        threads = [threading.Thread(target=run, args=w) for w in work]
        for t in threads:
            t.start()
        gate.wait()
        start = time.perf_counter()
        gate.wait()
        took = time.perf_counter() - start
        for t in threads:
            t.join()
        return took
    with D.Context() as a, D.Context() as b, D.Context() as c:
        assert min(seconds([a, b, c]) for _ in range(2)) <= 10 * min(seconds([a]) for _ in range(2))


def test_two_contexts_at_once(ctx):
    """Each has places of its own for the sums that its workgroups exchange."""
    shape = (8, 16, 104, 104)
    x, rm, rv, dp = _inputs(shape, 10)
    nan = np.full_like(x, np.nan)
    _, want = _run(ctx, shape, 10)
    with D.Context() as other:
        both = []
        for c in (ctx, other):
            m = _Place(c, 0, x=x, y=nan, p=np.full_like(dp, np.nan), rm=rm, rv=rv, sm=rm * 0, sv=rm * 0, dp=dp, t=nan, dz=nan)
            both.append((c, m, sum(_commands(m, shape), [])))
        for _ in range(20):
            for c, m, cmds in both:
                c.h2d(m["rm"], rm)
                c.h2d(m["rv"], rv)
                c.submit(cmds)
        for c, m, cmds in both:
            c.sync()
            got = m.all()
            for k in want:
                assert_bits_equal(got[k], want[k])


def _remade(fwd, bwd):
    fwd[0].flags |= _ffi.FLAG_BN_REMADE
    bwd[0].flags |= _ffi.FLAG_BN_REMADE
    return fwd, bwd


@pytest.mark.parametrize("polls", [None, 0, 1])
@pytest.mark.parametrize("shape", SHAPES)
def test_values_that_are_not_stored(ctx, shape, polls, monkeypatch):
    """GH_FLAG_BN_REMADE: what is still written has the bits of the commands without it, whatever lay in y's place; "t" as the
    gradient's place is no pair of one launch, so that the values are made again by a kernel of their own."""
    for dz in ("dz", "y", "t"):
        _, want = _run(ctx, shape, 12, dz=dz)
        if polls is not None:
            monkeypatch.setenv("GORGONIA_HIP_BN_POLLS", str(polls))
        with monkeypatch.context() as p:
            p.setitem(globals(), "_commands", lambda *a, plain=_commands, **kw: _remade(*plain(*a, **kw)))
            _, got = _run(ctx, shape, 12, dz=dz)
        monkeypatch.delenv("GORGONIA_HIP_BN_POLLS", raising=False)
        for k in ("x", "p", "sm", "sv", "rm", "rv", "dp", dz):
            assert_bits_equal(got[k], want[k], (dz, k))


def test_a_command_that_needs_the_one_behind_it(ctx):
    shape = (2, 3, 4, 4)
    x, rm, rv, dp = _inputs(shape, 13)
    m = _Place(ctx, 0, x=x, y=x, p=dp, rm=rm, rv=rv, sm=rm, sv=rv, dp=dp, t=x, dz=x)
    _, bwd = _remade(*_commands(m, shape))
    with pytest.raises(D.DeviceError):
        ctx.run(bwd[:1])
    ctx.clear_error()
    ctx.run(bwd)
    m.all()


@pytest.mark.parametrize("read", [None, "n", "dn"])
def test_on_a_tape(ctx, read):
    """A graph's normalised values are left out only where nobody else reads them: the same bits as operator by operator."""
    from gorgonia_amd import graph as G
    shape = (4, 16, 12, 12)
    x, rm0, rv0, dp = _inputs(shape, 14)

    def run(machine, **kw):
        g = G.NewGraph()
        z = G.LeakyRelu(G.NewTensor(g, x), 0.5)
        rm, rv, sm, sv = (G.NewTensor(g, v.copy(), resident=True) for v in (rm0, rv0, rm0 * 0, rm0 * 0))
        n = G.BatchNormTrain(z, rm, rv, sm, sv, momentum=MOMENTUM, epsilon=EPS)
        a = G.Rectify(n)
        p = G.MaxPool2D(a, (2, 2), (0, 0), (2, 2))
        dn = G.RectifyDiff(n, G.MaxPool2DDiff(a, G.HadamardProd(p, G.NewTensor(g, dp)), (2, 2), (0, 0), (2, 2)))
        dz = G.BatchNormDiff(z, dn, sm, sv, epsilon=EPS)
        out = {"dz": G.Read(dz), "p": G.Read(p), "rm": G.Read(rm), "rv": G.Read(rv)}
        if read:
            out[read] = G.Read({"n": n, "dn": dn}[read])
        m = machine(g, **kw)
        for _ in range(3):
            m.RunAll()
        got = {k: v.copy() for k, v in out.items()}
        m.Close()
        return got
    fused, apart = run(G.NewTapeMachine, fuse_activations=True), run(G.NewLispMachine)
    for k in apart:
        if k == "dz":   # two orders of adding the gradient's sums
            assert rel_frobenius(fused[k], apart[k].astype(np.float64)) <= U
        else:
            assert_bits_equal(fused[k], apart[k], k)
