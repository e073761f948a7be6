"""Uploads in pieces (gh_pieces.hip) whose copy does not begin: the kernels that wait copy the batch, and after the third such upload
the context's batches go whole.  Contexts whose streams may stand behind each other's."""
import threading
import time

import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.test_gpu_pieces import _Host
from tests.test_gpu_pieces_bits import DETECTOR, _Chain
from tests.util import assert_bits_equal

pytestmark = pytest.mark.gpu


class _Runs:
    """The front of a detector on a context of its own, and the results of the batch uploaded whole."""

    def __init__(self, ctx, monkeypatch, B=4):
        self.ctx, self.chain = ctx, _Chain(ctx, B, 416, 416, DETECTOR)
        self.host = _Host(ctx, self.chain.nbytes)
        self.host.fill(np.random.default_rng(B).uniform(0, 1, self.chain.shape).astype(np.float32))
        with monkeypatch.context() as p:
            p.setenv("GORGONIA_HIP_NO_PIECES", "1")
            self.want = self.chain.run(self.host.p)[0]

    def step(self):
        """Whether the batch went in pieces."""
        before = self.ctx.joint_launches(_ffi.JOINT_PIECES)[0]
        for g, w in zip(self.chain.run(self.host.p)[0], self.want):
            assert_bits_equal(g, w)
        return self.ctx.joint_launches(_ffi.JOINT_PIECES)[0] - before == 1

    def close(self):
        self.host.close()
        self.chain.close()


@pytest.mark.parametrize("ticks", [None, "0", "1000"])
def test_the_third_in_a_row_is_the_last(monkeypatch, ticks):
    with D.Context(0, 0) as ctx:
        runs = _Runs(ctx, monkeypatch)
        assert runs.step() and runs.step()
        with monkeypatch.context() as p:
            p.setenv("GORGONIA_HIP_PIECES_LATE", "1")
            if ticks:
                p.setenv("GORGONIA_HIP_PIECES_TICKS", ticks)
            assert [runs.step() for _ in range(5)] == [True, True, True, False, False]
        assert not runs.step()
        runs.close()


def test_two_now_and_then_are_not(monkeypatch):
    monkeypatch.setenv("GORGONIA_HIP_PIECES_TICKS", "0")
    with D.Context(0, 0) as ctx:
        runs = _Runs(ctx, monkeypatch, B=2)
        for _ in range(3):
            with monkeypatch.context() as p:
                p.setenv("GORGONIA_HIP_PIECES_LATE", "1")
                assert runs.step() and runs.step()
            for _ in range(65):   # (what is given up here counts not)
                assert runs.step()
        runs.close()


def test_contexts_side_by_side(monkeypatch):
    """More streams than hardware queues: whichever copies stand behind others' layers, every run ends with the
    whole batch's bits."""
    ctxs = [D.Context(0, 0) for _ in range(3)]
    runs = [_Runs(c, monkeypatch, B=2 + k) for k, c in enumerate(ctxs)]
    failed = []

    def work(r):
        try:
            for _ in range(8):
                r.step()
        except BaseException as e:   # noqa: BLE001 (told below)
            failed.append(e)
    threads = [threading.Thread(target=work, args=(r,)) for r in runs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
    for r in runs:
        r.close()
    for c in ctxs:
        c.close()


def test_given_up_once(monkeypatch):
    """Four pieces whose copy does not begin: one wait of a millisecond, not one of six for each."""
    with D.Context(0, 0) as ctx:
        runs = _Runs(ctx, monkeypatch, B=8)
        chain, took = runs.chain, []
        cmds = [D.cmd_copy(chain.x, runs.host.p.value, chain.nbytes)] + chain.layers
        monkeypatch.setenv("GORGONIA_HIP_PIECES_LATE", "1")
        for _ in range(3):
            t = time.perf_counter()
            ctx.submit(cmds)
            ctx.sync()
            took.append(time.perf_counter() - t)
        print("given up, ms:", [round(1e3 * t, 2) for t in took], flush=True)
        assert ctx.joint_launches(_ffi.JOINT_PIECES) == (3, 405)
        assert min(took) < 15e-3
        runs.close()


def test_a_message_names_the_callers_command(monkeypatch):
    """Behind the commands that ran in pieces, as where the batch went whole."""
    with D.Context(0, 0) as ctx:
        runs = _Runs(ctx, monkeypatch, B=2)
        chain = runs.chain
        cmds = [D.cmd_copy(chain.x, runs.host.p.value, chain.nbytes)] + chain.layers
        for at in (len(cmds), len(cmds) + 1):
            bad = cmds + [D.cmd_relu(chain.x, chain.x, 16)] * (at - len(cmds)) + [D.cmd_relu(chain.x, 0, 16)]
            said = []
            for whole in (False, True):
                with monkeypatch.context() as p:
                    if whole:
                        p.setenv("GORGONIA_HIP_NO_PIECES", "1")
                    before = ctx.joint_launches(_ffi.JOINT_PIECES)[0]
                    with pytest.raises(D.DeviceError) as e:
                        ctx.submit(bad)
                    assert ctx.joint_launches(_ffi.JOINT_PIECES)[0] - before == (not whole)
                said.append(str(e.value))
                ctx.clear_error()
                ctx.sync()
            assert said[0] == said[1] and f"cmd {at}:" in said[0], said
        runs.close()
