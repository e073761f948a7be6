"""Float64 products with a short contraction on tiles staged in LDS (k_dgemm): both tile sizes, ragged edges, odd strides
and offsets, every transposition, batches, one and several k-tiles, against the float64 product."""
import ctypes as C

import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.util import rel_frobenius

pytestmark = pytest.mark.gpu

# m, n, k, batch: 64x64 tiles whole, ragged and odd; 128x128 tiles; one to three k-tiles of 8 or 16, whole and not
SHAPES = [(1024, 1024, 16, 1), (1001, 1003, 1, 1), (561, 1679, 17, 1), (560, 1680, 48, 1), (130, 900, 31, 16), (66, 258, 32, 24), (2049, 2111, 9, 1),
          (2048, 2048, 24, 1), (385, 129, 3, 96), (104, 936, 8, 24)]


@pytest.fixture(scope="module")
def ctx():
    c = D.Context(0, 0)
    yield c
    c.close()


@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("m,n,k,batch", SHAPES)
@pytest.mark.parametrize("offset", [0, 1])
def test_product(ctx, m, n, k, batch, ta, tb, offset):
    rng = np.random.default_rng(m + k)
    a, b = rng.standard_normal((batch, m, k)), rng.standard_normal((batch, k, n))
    x = np.ascontiguousarray(a.transpose(0, 2, 1) if ta else a)
    y = np.ascontiguousarray(b.transpose(0, 2, 1) if tb else b)
    buffers = [ctx.malloc(8 * (v.size + offset)) for v in (x, y)] + [ctx.malloc(8 * (batch * m * n + 1))]
    px, py, pc = buffers[0] + 8 * offset, buffers[1] + 8 * offset, buffers[2]
    ctx.h2d(px, x)
    ctx.h2d(py, y)
    ctx.h2d(pc, np.full(batch * m * n + 1, np.nan))
    cmd = D.cmd_gemm(px, py, pc, m, n, k, trans_a=ta, trans_b=tb, batch=batch, stride_a=m * k, stride_b=k * n, stride_c=m * n, dtype=_ffi.F64)
    if not (offset and k > 32):   # 16-byte loads are part of the choice there
        assert ctx.lib.gh_runs_straight(C.byref(cmd)) == 0
    ctx.run(cmd)
    got = ctx.d2h(pc, (batch * m * n + 1,), np.float64)
    for p in buffers:
        ctx.free(p)
    assert np.isnan(got[-1])
    # sums of at most 48 products in the operands' own precision
    assert rel_frobenius(got[:-1].reshape(batch, m, n), a @ b) <= 1e-14
