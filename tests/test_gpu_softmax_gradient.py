"""A SoftMax, alone or in a product's epilogue, with the scaled tensor and the SoftMax gradient behind it in one launch (k_pairs.hip,
k_gemm.hip): the bits of the three commands submitted apart, in every tensor they write."""
import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.test_gpu_pairs import _Memory
from tests.util import assert_bits_equal

pytestmark = pytest.mark.gpu


def _check(ctx, commands, *arrays, form, shift=0):
    """commands(pointers) -> three commands; `form` of the launch that takes them (0: none does)."""
    out = []
    for together in (True, False):
        m = _Memory(ctx, *arrays, shift=shift)
        before = ctx.joint_launches(_ffi.JOINT_SOFTMAX_GRADIENT)[0]
        c = commands(m.ptr)
        if together:
            ctx.run(c)
        else:
            for k in c:
                ctx.run([k])
        after, seen = ctx.joint_launches(_ffi.JOINT_SOFTMAX_GRADIENT)
        assert after - before == (1 if together and form else 0)
        assert not (together and form) or seen == form
        out.append(m.all())
    assert_bits_equal(*out)


def _labels(rng, rows, cols, dt):
    x = np.zeros((rows, cols), dt)
    x[np.arange(rows), rng.integers(0, cols, rows)] = 1
    x[0, 0] = -0.0
    return x


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("where", ["apart", "in_place", "over_logits"])
@pytest.mark.parametrize("rows,cols", [(1, 1), (50, 10), (3, 63), (5, 64), (5, 65), (1031, 7)])
def test_behind_a_softmax(ctx, rows, cols, where, dt):
    rng = np.random.default_rng(rows + cols)
    code = _ffi.F32 if dt == np.float32 else _ffi.F64
    z = (rng.standard_normal((rows, cols)) * 4).astype(dt)
    if rows > 2:
        z[1, 0], z[2, cols - 1] = np.inf, np.nan
        z[rows - 1, :] = -np.inf
    none = np.full((rows, cols), np.nan, dt)

    def commands(q):
        y = q[0] if where == "in_place" else q[1]
        g = q[2] if where == "in_place" else q[4]
        return [D.cmd_softmax(q[0], y, rows, cols, dtype=code), D.cmd_bin("mul", "vs", q[2], q[3], z.size, dtype=code, dst=g),
                D.cmd_softmax_bwd(y, g, q[0] if where == "over_logits" else q[5], rows, cols, dtype=code)]
    _check(ctx, commands, z, none, _labels(rng, rows, cols, dt), np.array([-1.0 / 500], dt), none, none, form=1 if cols <= 64 else 0, shift=1)


# the 16-row kernel with eight and sixteen wavefronts, with rows that two tiles have; the slabs' sum, of few and of many rows;
# the kernels that do not take the three: 32-row tiles, and more than 16 columns in one piece
@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("M,N,K,bias,act,form", [(128, 10, 625, False, None, 2), (16, 16, 511, True, "relu", 2), (17, 1, 512, False, None, 2), (131, 7, 40, True, "leaky", 2),
                                                 (8, 10, 21632, False, None, 3), (15, 32, 4096, True, None, 3), (40, 10, 8192, False, "relu", 3),
                                                 (8, 10, 640, False, None, 0), (64, 24, 640, False, None, 0)])
def test_behind_a_product(ctx, M, N, K, bias, act, form, in_place):
    rng = np.random.default_rng(M + N + K)
    dt = np.float32
    a, b = rng.standard_normal((M, K)).astype(dt), (rng.standard_normal((K, N)) / np.sqrt(K)).astype(dt)
    none = np.full((M, N), np.nan, dt)

    def commands(q):
        g = q[4] if in_place else q[6]
        return [D.cmd_gemm(q[0], q[1], q[2], M, N, K, softmax=True, bias=q[3] if bias else 0, act=act, alpha=0.1),
                D.cmd_bin("mul", "vs", q[4], q[5], M * N, dst=g), D.cmd_softmax_bwd(q[2], g, q[7], M, N)]
    _check(ctx, commands, a, b, none, rng.standard_normal(N).astype(dt), _labels(rng, M, N, dt), np.array([-1.0 / 1280], dt), none, none, form=form)


def test_what_overlaps_runs_apart(ctx):
    """A gradient over what other workgroups of the product still read, or values that one launch could not see in order."""
    rng = np.random.default_rng(3)
    M, N, K = 64, 8, 64
    a, b, none = (rng.standard_normal(s).astype(np.float32) for s in ((M, K), (K, N), (M, N)))
    x, s = _labels(rng, M, N, np.float32), np.array([-0.25], np.float32)

    def of(dx, labels=3, y=None, rows=M):
        def commands(q):
            return [D.cmd_gemm(q[0], q[1], q[2], M, N, K, softmax=True), D.cmd_bin("mul", "vs", q[labels], q[4], rows * N, dst=q[5]),
                    D.cmd_softmax_bwd(q[2] if y is None else q[y], q[5], q[dx], rows, N)]
        return commands
    for commands in (of(0), of(1), of(6, labels=2), of(6, y=7), of(6, rows=M // 2)):
        _check(ctx, commands, a, b, none, x, s, none, none, none, form=0)
