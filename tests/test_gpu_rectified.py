"""A product and its Rectify, and a dense layer's two gradients with the Rectify's gradient behind them, in one launch (k_gemm.hip,
k_gemm_gradients.hip): the bits of the commands submitted apart, in every tensor they write."""
import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.test_gpu_pairs import _Memory
from tests.util import assert_bits_equal

pytestmark = pytest.mark.gpu


def _check(ctx, commands, *arrays, form, shift=0):
    """form of the launch that takes the Rectify along; None: none does."""
    out = []
    for together in (True, False):
        m = _Memory(ctx, *arrays, shift=shift)
        before = ctx.joint_launches(_ffi.JOINT_RECTIFIED)[0]
        for c in ([commands(m.ptr)] if together else [[k] for k in commands(m.ptr)]):
            ctx.run(c)
        after, seen = ctx.joint_launches(_ffi.JOINT_RECTIFIED)
        assert after - before == (1 if together and form is not None else 0)
        assert not (together and form is not None) or seen == form
        out.append(m.all())
    assert_bits_equal(*out)


# both tile widths with eight and sixteen wavefronts; rows and columns that two tiles have; float64 with an odd and an even K, and
# products that other kernels keep (32-row tiles, a product cut along K, tiled and direct ones)
@pytest.mark.parametrize("dt,M,N,K,form", [
    (np.float32, 128, 625, 1152, 36), (np.float32, 33, 50, 600, 26), (np.float32, 17, 100, 64, 18), (np.float32, 128, 700, 40, 28), (np.float32, 40, 7, 33, 18),
    (np.float32, 8, 625, 1152, None), (np.float32, 36, 40, 8192, None), (np.float32, 512, 1024, 512, None),
    (np.float64, 50, 625, 1152, 108), (np.float64, 19, 33, 77, 104), (np.float64, 7, 65, 301, 108), (np.float64, 640, 640, 640, None)])
@pytest.mark.parametrize("shift", [0, 1])
def test_product_and_rectify(ctx, dt, M, N, K, form, shift):
    rng = np.random.default_rng(M + N + K)
    code = _ffi.F64 if dt == np.float64 else _ffi.F32
    a, b, none = rng.standard_normal((M, K)).astype(dt), rng.standard_normal((K, N)).astype(dt), np.full((M, N), np.nan, dt)
    a[0, 0], a[M - 1, 0] = np.inf, np.nan
    b[:, N - 1] = 0
    _check(ctx, lambda q: [D.cmd_gemm(q[0], q[1], q[2], M, N, K, dtype=code), D.cmd_relu(q[2], q[3], M * N, dtype=code)], a, b, none, none, form=form, shift=shift)


# batch, inputs, outputs and whether the gradients are one launch: the small-output and the direct kernels as the input gradient's,
# float64's direct one beside a weight gradient of eight wavefronts; two launches
@pytest.mark.parametrize("dt,B,I,O,joint", [
    (np.float32, 128, 625, 10, True), (np.float32, 128, 1152, 625, True), (np.float32, 64, 300, 100, True), (np.float32, 33, 77, 50, True), (np.float32, 257, 54, 1536, True),
    (np.float64, 50, 625, 10, True), (np.float64, 50, 1152, 625, True), (np.float64, 96, 65, 33, True), (np.float64, 682, 296, 610, True), (np.float64, 1448, 96, 1582, True),
    (np.float64, 1448, 96, 200, False)])
@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("input_first", [False, True])
def test_gradients_and_rectify_gradient(ctx, dt, B, I, O, joint, in_place, input_first):
    rng = np.random.default_rng(B + I + O)
    code = _ffi.F64 if dt == np.float64 else _ffi.F32
    x, dy, w, z = (rng.standard_normal(s).astype(dt) for s in ((B, I), (B, O), (I, O), (B, I)))
    z.reshape(-1)[:5] = [0.0, -0.0, np.nan, np.inf, -np.inf]
    dw, dx, dz = (np.full(s, np.nan, dt) for s in ((I, O), (B, I), (B, I)))

    def commands(q):
        pair = [D.cmd_gemm(q[0], q[1], q[4], I, O, B, trans_a=True, dtype=code), D.cmd_gemm(q[1], q[2], q[5], B, I, O, trans_b=True, dtype=code)]
        return (pair[::-1] if input_first else pair) + [D.cmd_relu_bwd(q[3], q[5], q[5] if in_place else q[6], B * I, dtype=code)]
    before = ctx.joint_launches(_ffi.JOINT_DENSE_GRADIENTS)[0]
    m = _Memory(ctx, x, dy, w, z, dw, dx, dz)
    ctx.run(commands(m.ptr))
    m.all()
    launches, form = ctx.joint_launches(_ffi.JOINT_DENSE_GRADIENTS)
    assert launches - before == joint
    if B == 682:
        assert form == 1008010000   # (as in test_gpu_dense_gradients.py)
    _check(ctx, commands, x, dy, w, z, dw, dx, dz, form=0 if joint else None)


def test_what_overlaps_runs_apart(ctx):
    """Results over what the products still read, of another size, or of another tensor: as submitted apart."""
    rng = np.random.default_rng(7)
    B, I, O = 64, 96, 96
    x, dy, w, z = (rng.standard_normal(s).astype(np.float32) for s in ((B, I), (B, O), (I, O), (B, I)))
    dw, dx, dz = (np.full(s, np.nan, np.float32) for s in ((I, O), (B, I), (B, I)))

    def gradients(z_at=3, out=6, n=B * I):
        return lambda q: [D.cmd_gemm(q[0], q[1], q[4], I, O, B, trans_a=True), D.cmd_gemm(q[1], q[2], q[5], B, I, O, trans_b=True), D.cmd_relu_bwd(q[z_at], q[5], q[out], n)]

    def forward(out, n=B * O, src=5):
        return lambda q: [D.cmd_gemm(q[0], q[2], q[5], B, O, I), D.cmd_relu(q[src], q[out], n)]
    for commands in (gradients(out=0), gradients(out=1), gradients(z_at=4), gradients(z_at=5), gradients(out=3), gradients(n=B * I - 1), forward(5), forward(0), forward(2),
                     forward(6, n=B * O // 2), forward(6, src=3)):
        _check(ctx, commands, x, dy, w, z, dw, dx, dz, form=None)
