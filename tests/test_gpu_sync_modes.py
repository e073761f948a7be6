"""How gh_sync waits (GORGONIA_HIP_SYNC, read when a context is made): the numbers are there in every mode, and a spinning
wait keeps the thread busy to its end."""
import time

import numpy as np
import pytest

from gorgonia_amd import device as D

pytestmark = pytest.mark.gpu


def _share_of_the_wait_spent_computing(n=2048, products=120):
    ctx = D.Context(0, 0)
    a = np.random.default_rng(0).integers(-3, 4, (n, n)).astype(np.float32)
    pa, pc = ctx.upload(a), ctx.malloc(a.nbytes)
    cmds = [D.cmd_gemm(pa, pa, pc, n, n, n)] * products
    ctx.run(cmds[:2])
    shares = []
    for _ in range(3):
        ctx.submit(cmds)
        wall, own = time.perf_counter(), time.thread_time()
        ctx.sync()
        wall, own = time.perf_counter() - wall, time.thread_time() - own
        assert wall > 0.005
        shares.append(own / wall)
    assert np.array_equal(ctx.d2h(pc, a.shape), (a.astype(np.float64) @ a).astype(np.float32))
    for _ in range(70):   # waits of a few microseconds, some of them in the runtime
        ctx.run(cmds[0])
    ctx.free(pa)
    ctx.free(pc)
    ctx.close()
    return max(shares)


@pytest.mark.parametrize("mode", [None, "block", "spin"])
def test_modes(monkeypatch, mode):
    if mode:
        monkeypatch.setenv("GORGONIA_HIP_SYNC", mode)
    else:
        monkeypatch.delenv("GORGONIA_HIP_SYNC", raising=False)
    share = _share_of_the_wait_spent_computing()
    assert share > 0.9 or mode != "spin"   # (what the runtime's own wait does in the other modes is its affair)
