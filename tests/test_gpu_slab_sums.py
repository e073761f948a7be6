"""Sums of filter-gradient slabs that wait for the commands behind them (k_slab_sums.hip): the bits of one submission for each
command, also where a command behind the gradient reads or overwrites its result."""
import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.util import assert_bits_equal

pytestmark = pytest.mark.gpu


class _Tensors:
    def __init__(self, ctx, dt):
        self.ctx, self.dt, self.rng, self.all = ctx, dt, np.random.default_rng(4), []

    def make(self, *shape):
        p = self.ctx.upload(self.rng.standard_normal(shape).astype(self.dt))
        self.all.append((p, shape))
        return p

    def values(self):
        out = [self.ctx.d2h(p, shape, self.dt) for p, shape in self.all]
        for p, _ in self.all:
            self.ctx.free(p)
        return out


def _same(ctx, build, dt=np.float32):
    got = []
    for together in (True, False):
        t = _Tensors(ctx, dt)
        cmds = build(t)
        for group in ([cmds] if together else [[c] for c in cmds]):
            ctx.run(group)
        got.append(t.values())
    for a, b in zip(*got):
        assert_bits_equal(a, b)


# B, C, H, W, F: slabs summed by groups of 64 and of 16 results, by lanes from the small-image and the single-channel kernel
# (64 slabs and fewer) and from the vector kernel, one after the other from the tiled kernel
LAYERS = [(8, 64, 26, 26, 128), (8, 16, 52, 52, 32), (64, 32, 14, 14, 64), (16, 64, 7, 7, 128), (64, 1, 28, 28, 32), (5, 1, 20, 20, 8), (6, 2, 12, 12, 8), (2, 150, 9, 9, 140)]


def _gradient(t, layer, dt=_ffi.F32, dw=None):
    B, C, H, W, F = layer
    return D.cmd_conv2d_bwd_filter(t.make(B, C, H, W), t.make(B, F, H, W), dw or t.make(F, C, 3, 3), B, C, H, W, F, 3, 3, pad=(1, 1), dtype=dt)


@pytest.mark.parametrize("code,np_dt", [(_ffi.F32, np.float32), (_ffi.F64, np.float64)])
def test_gradients_one_behind_the_other(ctx, code, np_dt):
    """More of them than one launch sums."""
    _same(ctx, lambda t: [_gradient(t, layer, code) for layer in LAYERS + LAYERS[:4]], np_dt)


def test_a_backward_pass_and_its_solver(ctx):
    def build(t):
        cmds, weights = [], []
        for B, C, H, W, F in ((4, 32, 26, 26, 64), (4, 16, 52, 52, 32)):
            x, dy, w, dw, dx = t.make(B, C, H, W), t.make(B, F, H, W), t.make(F, C, 3, 3), t.make(F, C, 3, 3), t.make(B, C, H, W)
            cmds += [D.cmd_conv2d_bwd_filter(x, dy, dw, B, C, H, W, F, 3, 3, pad=(1, 1)), D.cmd_conv2d_bwd_data(dy, w, dx, B, C, H, W, F, 3, 3, pad=(1, 1)),
                     D.cmd_maxpool2d_bwd(x, t.make(B, C, H // 2, W // 2), dx, B, C, H, W, 2, 2, (0, 0), (2, 2))]
            weights.append((w, dw, F * C * 9))
        return cmds + [D.cmd_solver_step("vanilla", w, dw, n, (0.01,) + (0.0,) * 9, 0) for w, dw, n in weights]
    _same(ctx, build)


def test_a_result_that_the_next_command_reads_or_writes(ctx):
    layer = (8, 16, 52, 52, 32)
    B, C, H, W, F = layer

    def read(t):   # as the filters of the image gradient behind it
        g = _gradient(t, layer)
        return [g, D.cmd_conv2d_bwd_data(t.make(B, F, H, W), g.ptr[2], t.make(B, C, H, W), B, C, H, W, F, 3, 3, pad=(1, 1))]

    def inside(t):   # a flat buffer of gradients, of which a pooling gradient overwrites the middle
        flat = t.make(3 * F * C * 9)
        item = 4
        return [_gradient(t, layer, dw=flat), _gradient(t, layer, dw=flat + item * 2 * F * C * 9),
                D.cmd_maxpool2d_bwd(t.make(1, 1, 32, 32), t.make(1, 1, 16, 16), flat + item * (F * C * 9 - 500), 1, 1, 32, 32, 2, 2, (0, 0), (2, 2))]

    def twice(t):   # the same result again
        g = _gradient(t, layer)
        return [g, _gradient(t, layer, dw=g.ptr[2])]

    def elsewhere(t):   # a command of another kind
        g = _gradient(t, layer)
        return [g, D.cmd_relu(g.ptr[2], t.make(F, C, 3, 3), F * C * 9)]

    for build in (read, inside, twice, elsewhere):
        _same(ctx, build)


@pytest.mark.parametrize("code,np_dt", [(_ffi.F32, np.float32), (_ffi.F64, np.float64)])
@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("member", [1, 2])
def test_a_result_inside_a_run_of_elementwise_commands(ctx, code, np_dt, in_place, member):
    """The run's first command has nothing to do with the result; its second or third reads it, or writes over it."""
    layer = (64, 32, 14, 14, 64)
    n = 64 * 32 * 9
    counts = []

    def build(t):
        g = _gradient(t, layer, code)
        run = [D.cmd_relu_bwd(t.make(n), t.make(n), t.make(n), n, dtype=code)]
        if member == 2:
            run.append(D.cmd_relu(t.make(n), t.make(n), n, dtype=code))
        run.append(D.cmd_relu(g.ptr[2], g.ptr[2] if in_place else t.make(n), n, dtype=code))
        counts.append(_ffi.load().gh_elementwise_run((_ffi.GhCmd * len(run))(*run), len(run)))
        return [g] + run
    _same(ctx, build, np_dt)
    assert counts[0] == member + 1   # one run


def test_replays(ctx):
    layer = (8, 16, 52, 52, 32)
    t = _Tensors(ctx, np.float32)
    cmds = [_gradient(t, layer), _gradient(t, (8, 64, 26, 26, 128))]
    ctx.run(cmds)
    want = [ctx.d2h(p, shape, np.float32) for p, shape in t.all]
    ctx.graph_begin()
    ctx.submit(cmds)
    graph = ctx.graph_end()
    for _ in range(3):
        for p, shape in (t.all[2], t.all[5]):
            ctx.h2d(p, np.full(shape, np.nan, np.float32))
        ctx.graph_launch(graph)
        ctx.sync()
        for (p, shape), w in zip(t.all, want):
            assert_bits_equal(ctx.d2h(p, shape, np.float32), w)
        ctx.run(cmds[:1])
    ctx.graph_destroy(graph)
    t.values()
