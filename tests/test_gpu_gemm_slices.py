"""Small-output products whose long contraction is cut into slices: the edges of the cut, every epilogue, both
kernels, against float64 products."""
import ctypes as C

import numpy as np
import pytest

from gorgonia_amd import device as D
from tests.util import rel_frobenius

pytestmark = pytest.mark.gpu

# m, n, k: one tile and few, rows below and above sixteen (up to four of wide products run elsewhere), k one below and at the first cut, ragged, not a multiple of
# the slices' chunks, so long that the device is full
SHAPES = [(8, 10, 21632), (9, 300, 2048), (1, 1, 2047), (20, 30, 4001), (64, 10, 4096), (16, 16, 2048), (33, 32, 2500), (7, 45, 5003),
          (100, 17, 3333), (512, 32, 2064)]


@pytest.fixture(scope="module")
def ctx():
    c = D.Context(0, 0)
    yield c
    c.close()


def _product(ctx, a, b, m, n, k, **kw):
    pa, pb, pc = ctx.upload(a), ctx.upload(b), ctx.upload(np.full((m, n), np.nan, np.float32))
    bias = kw.pop("bias", None)
    if bias is not None:
        kw["bias"] = ctx.upload(bias)
    cmd = D.cmd_gemm(pa, pb, pc, m, n, k, **kw)
    ctx.run(cmd)
    got = ctx.d2h(pc, (m, n))
    ctx.run(cmd)
    assert np.array_equal(got, ctx.d2h(pc, (m, n)))
    slices = C.c_int()
    ctx.lib.gh_gemm_route(C.byref(cmd), C.byref(slices))
    for p in (pa, pb, pc) + ((kw["bias"],) if bias is not None else ()):
        ctx.free(p)
    return got, slices.value


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_product(ctx, m, n, k):
    rng = np.random.default_rng(k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    want = a.astype(np.float64) @ b
    got, slices = _product(ctx, a, b, m, n, k)
    assert (slices > 1) == (k >= 2048)
    assert rel_frobenius(got, want) <= 1e-5
    if m >= 16:
        for kw, x, y in (({"trans_a": True}, a.T, b), ({"trans_b": True}, a, b.T)):
            got, _ = _product(ctx, np.ascontiguousarray(x), np.ascontiguousarray(y), m, n, k, **kw)
            assert rel_frobenius(got, want) <= 1e-5


@pytest.mark.parametrize("m,n,k", [s for s in SHAPES if s[1] <= 32])
def test_epilogues_are_those_of_the_separate_operators(ctx, m, n, k):
    rng = np.random.default_rng(k + 1)
    a, b = rng.uniform(-1, 1, (m, k)).astype(np.float32), (rng.uniform(-1, 1, (k, n)) / 64).astype(np.float32)
    bias = rng.uniform(-1, 1, (n,)).astype(np.float32)
    bare, _ = _product(ctx, a, b, m, n, k)
    z = bare + bias
    z = z * (z >= 0)
    got, _ = _product(ctx, a, b, m, n, k, bias=bias, act="relu")
    assert np.array_equal(got, z)
    pz, py = ctx.upload(z), ctx.malloc(z.nbytes)
    ctx.run(D.cmd_softmax(pz, py, m, n))
    want = ctx.d2h(py, z.shape)
    ctx.free(pz), ctx.free(py)
    got, _ = _product(ctx, a, b, m, n, k, bias=bias, act="relu", softmax=True)
    assert np.array_equal(got, want)
