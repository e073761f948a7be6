"""A batch out of pinned host memory in pieces, the layers behind it piece by piece (gh_pieces.hip): the bits of the same
commands on each piece's images, submitted one by one."""
import ctypes as C

import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D

pytestmark = pytest.mark.gpu

PIECE = 4 << 20


class _Net:
    """An upload, two convolutions with a pooling between them and, not in pieces, a copy of what they made."""

    def __init__(self, ctx, B, H, W, together=False):
        self.ctx, self.B, self.H, self.W = ctx, B, H, W
        r = np.random.default_rng(B + H)
        self.nbytes, self.F, self.ph, self.pw = 12 * B * H * W, 8, (H - 2) // 2 + 1, (W - 2) // 2 + 1
        self.n = (B * self.F * H * W, B * self.F * self.ph * self.pw, B * 16 * self.ph * self.pw)
        self.w = [ctx.upload(r.standard_normal(s).astype(np.float32)) for s in ((self.F, 3, 3, 3), (16, self.F, 3, 3))]
        self.x = ctx.malloc(max(self.nbytes, 4 * self.n[1]))
        # the pooled values in the batch's own memory: the pieces end in front of the pooling
        self.y = [ctx.malloc(4 * self.n[0]), self.x if together else ctx.malloc(4 * self.n[1]), ctx.malloc(4 * self.n[2])]
        self.copy = ctx.malloc(4 * self.n[2])

    def layers(self, first, images):
        px, (p0, p1, p2) = self.x + first * (self.nbytes // self.B), [y + first * 4 * (n // self.B) for y, n in zip(self.y, self.n)]
        H, W, F, ph, pw = self.H, self.W, self.F, self.ph, self.pw
        return [D.cmd_conv2d(px, self.w[0], p0, images, 3, H, W, F, 3, 3, (1, 1)),
                D.cmd_maxpool2d(p0, p1, images, F, H, W, 2, 2, (0, 0, 0, 0), (2, 2)),
                D.cmd_conv2d(p1, self.w[1], p2, images, F, ph, pw, 16, 3, 3, (1, 1))]

    def submit(self, host):
        self.ctx.submit([D.cmd_copy(self.x, host.value, self.nbytes)] + self.layers(0, self.B) + [D.cmd_copy(self.copy, self.y[2], 4 * self.n[2])])

    def result(self):
        return self.ctx.d2h(self.copy, (self.n[2],))

    def one_by_one(self, x, pieces, head):
        self.ctx.h2d(self.x, x)
        ends = [0] + [(self.B * (p + 1) + pieces - 1) // pieces for p in range(pieces)]
        for a, b in zip(ends, ends[1:]):
            for c in self.layers(a, b - a)[:head]:
                self.ctx.run([c])
        for c in self.layers(0, self.B)[head:]:
            self.ctx.run([c])
        return self.ctx.d2h(self.y[2], (self.n[2],))

    def close(self):
        for p in {*self.w, self.x, *self.y, self.copy}:
            self.ctx.free(p)


class _Host:
    def __init__(self, ctx, nbytes):
        self.ctx, self.p = ctx, C.c_void_p()
        ctx.check(ctx.lib.gh_host_alloc(ctx.h, nbytes, C.byref(self.p)))

    def fill(self, x):
        C.memmove(self.p, x.ctypes.data, x.nbytes)
        return self.p

    def close(self):
        self.ctx.check(self.ctx.lib.gh_host_free(self.ctx.h, self.p))


# two images, fewer images than pieces would be, a piece of more than the last, images and a batch that are no multiple of 16
# bytes, and pieces that something else than the copy's workgroups copies, in part or altogether
@pytest.mark.parametrize("ticks", [None, "0", "300"])
@pytest.mark.parametrize("B,H,W", [(2, 416, 416), (3, 512, 480), (5, 271, 271), (8, 416, 416), (33, 111, 113)])
def test_pieces(ctx, monkeypatch, B, H, W, ticks):
    if ticks is not None:
        monkeypatch.setenv("GORGONIA_HIP_PIECES_TICKS", ticks)
    net = _Net(ctx, B, H, W)
    hosts = [_Host(ctx, net.nbytes) for _ in range(2)]
    count = min(B, 8, max(2, -(-net.nbytes // PIECE)))
    before, seen = ctx.joint_launches(_ffi.JOINT_PIECES)[0], []
    for step in range(3):
        xs = [np.random.default_rng(2 * step + k).standard_normal(net.nbytes // 4).astype(np.float32) for k in range(2)]
        for host, x in zip(hosts, xs):   # the second behind the first, without a wait between them
            net.submit(host.fill(x))
        ctx.sync()
        seen.append((xs[1], net.result()))
    launches, form = ctx.joint_launches(_ffi.JOINT_PIECES)
    assert launches - before == 6 and form == 100 * count + 3, (launches - before, form)
    for x, got in seen:
        assert np.array_equal(net.one_by_one(x, count, form % 100).view(np.uint32), got.view(np.uint32))
    for h in hosts:
        h.close()
    net.close()


def test_values_that_lie_together(ctx):
    net, host = _Net(ctx, 8, 416, 416, together=True), None
    host = _Host(ctx, net.nbytes)
    x = np.random.default_rng(0).standard_normal(net.nbytes // 4).astype(np.float32)
    net.submit(host.fill(x))
    ctx.sync()
    got, form = net.result(), ctx.joint_launches(_ffi.JOINT_PIECES)[1]
    assert form % 100 == 1, form
    assert np.array_equal(net.one_by_one(x, form // 100, 1).view(np.uint32), got.view(np.uint32))
    host.close()
    net.close()


def test_under_capture(ctx):
    """Recorded as the whole commands: a replay reads what lies in the pinned memory then."""
    net = _Net(ctx, 4, 416, 416)
    host = _Host(ctx, net.nbytes)
    before = ctx.joint_launches(_ffi.JOINT_PIECES)[0]
    ctx.graph_begin()
    net.submit(host.p)
    graph = ctx.graph_end()
    for step in range(3):
        x = np.random.default_rng(step).standard_normal(net.nbytes // 4).astype(np.float32)
        host.fill(x)
        ctx.graph_launch(graph)
        ctx.sync()
        got = net.result()
        assert np.array_equal(net.one_by_one(x, 1, 3).view(np.uint32), got.view(np.uint32))
    assert ctx.joint_launches(_ffi.JOINT_PIECES)[0] == before
    ctx.graph_destroy(graph)
    host.close()
    net.close()
