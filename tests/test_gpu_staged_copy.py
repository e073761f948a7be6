"""gh_memcpy_staged: a kernel that follows the host's copy into pinned memory; every byte, and none besides."""
import ctypes as C

import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D

pytestmark = pytest.mark.gpu

FROM, RANGE = 128 << 10, 16384
GUARD = 64


class _Stage:
    def __init__(self, ctx, nbytes):
        self.ctx, self.p = ctx, C.c_void_p()
        ctx.check(ctx.lib.gh_host_alloc(ctx.h, nbytes, C.byref(self.p)))

    def __enter__(self):
        return self.p

    def __exit__(self, *a):
        self.ctx.sync()
        self.ctx.check(self.ctx.lib.gh_host_free(self.ctx.h, self.p))


def _copy(ctx, nbytes, shift=0, passes=2):
    """nbytes to `shift` bytes behind an aligned address, fresh values in each pass, the bytes around them untouched."""
    words = nbytes // 4
    base = ctx.malloc(nbytes + shift + 4 * GUARD)
    with _Stage(ctx, nbytes) as stage:
        for p in range(passes):
            src = np.random.default_rng(p).integers(0, 2 ** 32, words, dtype=np.uint32)
            around = np.full((nbytes + shift) // 4 + GUARD, 0xA5A5A5A5, np.uint32)
            ctx.h2d(base, around)
            ctx.check(ctx.lib.gh_memcpy_staged(ctx.h, base + shift, stage, src.ctypes.data, nbytes))
            ctx.sync()
            around[shift // 4:shift // 4 + words] = src
            assert np.array_equal(ctx.d2h(base, around.shape, np.uint32), around)
    ctx.free(base)


# both sides of the size from which a kernel follows, whole ranges and parts of one, a last word alone, fewer ranges than
# workgroups and more, and a value that is copied in longer parts
@pytest.mark.parametrize("nbytes", [4, FROM - 4, FROM, FROM + 4, FROM + 12, 9 * RANGE + 16, 31 * RANGE + 4, 33 * RANGE, 2_076_672, 4_153_348, (14 << 20) + 20])
def test_every_byte(ctx, nbytes):
    _copy(ctx, nbytes)


@pytest.mark.parametrize("shift", [4, 8, 16])
def test_destinations(ctx, shift):
    _copy(ctx, 40 * RANGE + 8, shift=shift)


@pytest.mark.parametrize("ticks", ["0", "100"])
def test_a_kernel_that_does_not_wait(ctx, ticks, monkeypatch):
    """The kernel gives up before the host has said anything, the host's clock says so, and the value is copied again."""
    monkeypatch.setenv("GORGONIA_HIP_STAGED_TICKS", ticks)
    _copy(ctx, 2_076_672, passes=4)


def test_commands_behind_it_read_the_new_value(ctx):
    n = 300_000
    dst, out = ctx.malloc(4 * n), ctx.malloc(4 * n)
    with _Stage(ctx, 4 * n) as stage:
        for p in range(4):
            src = np.random.default_rng(p).standard_normal(n).astype(np.float32)
            ctx.check(ctx.lib.gh_memcpy_staged(ctx.h, dst, stage, src.ctypes.data, 4 * n))
            ctx.run([D.cmd_relu(dst, out, n)])
            assert np.array_equal(ctx.d2h(out, (n,)), np.maximum(src, 0))
    ctx.free(dst)
    ctx.free(out)


def test_under_capture(ctx):
    """Recorded as the copy out of the staging memory: a replay moves what lies there then."""
    n = 100_000
    dst = ctx.malloc(4 * n)
    src = np.arange(n, dtype=np.float32)
    with _Stage(ctx, 4 * n) as stage:
        ctx.graph_begin()
        ctx.check(ctx.lib.gh_memcpy_staged(ctx.h, dst, stage, src.ctypes.data, 4 * n))
        graph = ctx.graph_end()
        for p in range(3):
            now = src + p
            C.memmove(stage, now.ctypes.data, 4 * n)
            ctx.graph_launch(graph)
            ctx.sync()
            assert np.array_equal(ctx.d2h(dst, (n,)), now)
        ctx.graph_destroy(graph)
    ctx.free(dst)


def test_staging_memory_of_another_kind_is_refused(ctx):
    a = np.zeros(FROM, np.uint8)
    dst = ctx.malloc(FROM)
    assert ctx.lib.gh_memcpy_staged(ctx.h, dst, a.ctypes.data, a.ctypes.data, FROM) == _ffi.GH_EINVAL
    ctx.clear_error()
    ctx.free(dst)
