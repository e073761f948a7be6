"""Two commands in one launch (k_pairs.hip): the bits of the two commands submitted apart, every tensor they write."""
import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.util import assert_bits_equal

pytestmark = pytest.mark.gpu

SPECIAL = [0.0, -0.0, np.inf, -np.inf, np.nan, 5e-324, -5e-324, 1.7e308, -1.7e308]


def _values(rng, shape, dt=np.float64):
    x = np.round(rng.standard_normal(shape) * 2) / 2      # ties inside windows
    flat = x.reshape(-1)
    at = rng.integers(0, flat.size, min(9, flat.size))
    with np.errstate(over="ignore"):
        flat[at] = np.array(SPECIAL[:at.size], dt)
    return x.astype(dt)


class _Memory:
    """Tensors one after the other, `shift` elements from an aligned address."""

    def __init__(self, ctx, *arrays, shift=0):
        self.ctx, self.item, self.sizes, self.shapes, self.dt = ctx, arrays[0].itemsize, [], [a.shape for a in arrays], arrays[0].dtype
        flat = [np.full(shift, np.nan, self.dt)]
        self.at = []
        n = shift
        for a in arrays:
            self.at.append(n)
            pad = -a.size % 4
            flat += [a.ravel(), np.full(pad, np.nan, self.dt)]
            n += a.size + pad
        self.n, self.base = n, ctx.upload(np.concatenate(flat))
        self.ptr = [self.base + self.item * i for i in self.at]

    def all(self):
        out = self.ctx.d2h(self.base, (self.n,), self.dt)
        self.ctx.free(self.base)
        return out


def _both(ctx, commands, *arrays, shift=0):
    """commands(pointers) -> two commands; all memory behind one submit, and behind one submit each."""
    out = []
    for together in (True, False):
        m = _Memory(ctx, *arrays, shift=shift)
        c = commands(m.ptr)
        if together:
            ctx.run(c)
        else:
            ctx.run([c[0]])
            ctx.run([c[1]])
        out.append(m.all())
    assert_bits_equal(*out)


SHAPES = [(2, 3, 28, 28), (1, 1, 2, 2), (3, 2, 7, 7), (2, 5, 3, 8), (1, 4, 14, 5), (50, 32, 28, 28), (1, 1, 2, 3)]


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("B,C,H,W", SHAPES)
def test_rectify_and_pooling(ctx, B, C, H, W, in_place, shift):
    rng = np.random.default_rng(B + C + H + W)
    x = _values(rng, (B, C, H, W))
    a, p = np.full_like(x, np.nan), np.full((B, C, H // 2, W // 2), np.nan)

    def commands(q):
        to = q[0] if in_place else q[1]
        return [D.cmd_relu(q[0], to, x.size, dtype=_ffi.F64), D.cmd_maxpool2d(to, q[2], B, C, H, W, 2, 2, (0, 0, 0, 0), (2, 2), dtype=_ffi.F64)]
    _both(ctx, commands, x, a, p, shift=shift)


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("B,C,H,W", SHAPES)
def test_pooling_gradient_and_rectify_gradient(ctx, B, C, H, W, in_place, shift):
    rng = np.random.default_rng(B + C + H + W + 1)
    z = _values(rng, (B, C, H, W))
    with np.errstate(invalid="ignore"):
        a = z * (z >= 0)
    dy = _values(rng, (B, C, H // 2, W // 2))
    da, dz = np.full_like(z, np.nan), np.full_like(z, np.nan)

    def commands(q):
        return [D.cmd_maxpool2d_bwd(q[1], q[2], q[3], B, C, H, W, 2, 2, (0, 0, 0, 0), (2, 2), dtype=_ffi.F64),
                D.cmd_relu_bwd(q[0], q[3], q[3] if in_place else q[4], z.size, dtype=_ffi.F64)]
    _both(ctx, commands, z, a, dy, da, dz, shift=shift)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("rows,cols", [(1, 1), (128, 10), (50, 10), (3, 64), (5, 65), (2, 300), (1031, 7)])
def test_scaled_softmax_gradient(ctx, rows, cols, in_place, dt):
    rng = np.random.default_rng(rows + cols)
    code = _ffi.F32 if dt == np.float32 else _ffi.F64
    x, y = rng.standard_normal((rows, cols)).astype(dt), rng.random((rows, cols)).astype(dt)
    x.reshape(-1)[0] = -0.0
    s, t, dx = np.array([-1.0 / 1280], dt), np.full((rows, cols), np.nan, dt), np.full((rows, cols), np.nan, dt)

    def commands(q):
        g = q[0] if in_place else q[3]
        return [D.cmd_bin("mul", "vs", q[0], q[2], x.size, dtype=code, dst=g), D.cmd_softmax_bwd(q[1], g, q[4], rows, cols, dtype=code)]
    _both(ctx, commands, x, y, s, t, dx)


def test_what_overlaps_runs_apart(ctx):
    """The second command writes where the first one reads: one launch would race, and the result is the two commands'."""
    rng = np.random.default_rng(5)
    B, C, H, W = 2, 3, 8, 8
    z, a, dy, da = (_values(rng, (B, C, H, W)), _values(rng, (B, C, H, W)), _values(rng, (B, C, 4, 4)), np.full((B, C, H, W), np.nan))

    def over_input(q):      # dz over a, the pooling's input
        return [D.cmd_maxpool2d_bwd(q[1], q[2], q[3], B, C, H, W, 2, 2, (0, 0, 0, 0), (2, 2), dtype=_ffi.F64), D.cmd_relu_bwd(q[0], q[3], q[1], z.size, dtype=_ffi.F64)]

    def other_size(q):      # half of the tensor only
        return [D.cmd_maxpool2d_bwd(q[1], q[2], q[3], B, C, H, W, 2, 2, (0, 0, 0, 0), (2, 2), dtype=_ffi.F64), D.cmd_relu_bwd(q[0], q[3], q[3], z.size // 2, dtype=_ffi.F64)]

    def pool_over_x(q):     # the pooled values over the Rectify's input
        return [D.cmd_relu(q[0], q[1], z.size, dtype=_ffi.F64), D.cmd_maxpool2d(q[1], q[0], B, C, H, W, 2, 2, (0, 0, 0, 0), (2, 2), dtype=_ffi.F64)]

    def padded(q):
        return [D.cmd_relu(q[0], q[1], z.size, dtype=_ffi.F64), D.cmd_maxpool2d(q[1], q[3], B, C, H, W, 2, 2, (1, 0, 1, 0), (2, 2), dtype=_ffi.F64)]

    def dx_over_y(q):
        n = 24 * 16
        return [D.cmd_bin("mul", "vs", q[0], q[2], n, dtype=_ffi.F64, dst=q[3]), D.cmd_softmax_bwd(q[1], q[3], q[0], 24, 16, dtype=_ffi.F64)]
    for commands in (over_input, other_size, pool_over_x, padded, dx_over_y):
        _both(ctx, commands, z, a, dy, da)


def test_second_command_invalid(ctx):
    """The first command runs and the error is the second one's, as apart."""
    c = D.Context(0, 0)
    x = np.arange(-8, 8, dtype=np.float64)
    px, pa = c.upload(x), c.upload(np.zeros(16))
    bad = D.cmd_maxpool2d(pa, 0, 1, 1, 4, 4, 2, 2, (0, 0, 0, 0), (2, 2), dtype=_ffi.F64)
    with pytest.raises(D.DeviceError, match="cmd 1"):
        c.submit([D.cmd_relu(px, pa, 16, dtype=_ffi.F64), bad])
    c.close()
