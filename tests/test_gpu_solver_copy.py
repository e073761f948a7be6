"""A small copy behind a run of solver steps rides in their launch: the bits of the commands apart, also where the copy has to
do with what the steps write."""
import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.util import assert_bits_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("code,dt", [(_ffi.F32, np.float32), (_ffi.F64, np.float64)])
@pytest.mark.parametrize("kind,steps", [("vanilla", 1), ("rmsprop", 3), ("adam", 8)])
@pytest.mark.parametrize("src,dst,words", [("out", "host", 1), ("out", "host", 320), ("out", "host", 16384), ("out", "host", 16385), ("w", "host", 100), ("out", "g", 100), ("g", "host", 257)])
def test_copy_behind_solver_steps(ctx, code, dt, kind, steps, src, dst, words):
    n = 40_000
    par = {"vanilla": (0.01,) + (0.0,) * 9, "rmsprop": (0.01, 1e-8, 0, 1e-6, 5.0, 1.0, 0.9, 0.1, 0, 0), "adam": (0.001, 1e-8, 0, 0, 0, 1.0, 0.9, 0.999, 10.0, 31.0)}[kind]
    got = []
    for together in (True, False):
        rng = np.random.default_rng(words)
        t = {k: [ctx.upload(rng.uniform(0.1, 1.0, n).astype(dt)) for _ in range(steps)] for k in ("w", "g", "c1", "c2")}
        t["out"], t["host"] = [ctx.upload(rng.standard_normal(n).astype(dt))], [ctx.upload(np.zeros(n, dt))]
        cmds = [D.cmd_solver_step(kind, t["w"][i], t["g"][i], n - i, par, 0, t["c1"][i] if kind != "vanilla" else 0, t["c2"][i] if kind == "adam" else 0, dtype=code)
                for i in range(steps)]
        cmds.append(D.cmd_copy(t[dst][-1], t[src][-1], 4 * words))
        for group in ([cmds] if together else [[c] for c in cmds]):
            ctx.run(group)
        got.append([ctx.d2h(p, (n,), dt) for k in t for p in t[k]])
        for k in t:
            for p in t[k]:
                ctx.free(p)
    for a, b in zip(*got):
        assert_bits_equal(a, b)
