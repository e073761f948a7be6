"""A run of elementwise commands in one submit is executed in one pass: it has to store the bits the same
commands store when each is submitted by itself, in every tensor they name."""
import numpy as np
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D

pytestmark = pytest.mark.gpu

UNARY = sorted(_ffi.UNARY_FN)
BINARY = sorted(_ffi.BIN_FN)


@pytest.fixture(scope="module")
def ctx():
    c = D.Context(0, 0)
    yield c
    c.close()


def _both(ctx, make, tensors):
    """Every tensor after the commands in one submit, and after one submit per command."""
    got = []
    for together in (True, False):
        p = {k: ctx.upload(v) for k, v in tensors.items()}
        cmds = make(p)
        if together:
            ctx.run(cmds)
        else:
            for c in cmds:
                ctx.run(c)
        got.append({k: ctx.d2h(p[k], v.shape, v.dtype) for k, v in tensors.items()})
        for q in p.values():
            ctx.free(q)
    return got


def _same(got):
    for k in got[0]:
        a, b = got[0][k], got[1][k]
        bits = np.uint32 if a.dtype == np.float32 else np.uint64
        assert np.array_equal(a.view(bits), b.view(bits)), f"{k}: {np.sum(a.view(bits) != b.view(bits))} of {a.size} differ"


def _tensors(rng, shape, mid, np_dt):
    t = {k: rng.uniform(-3, 3, shape).astype(np_dt) for k in "abcd"}
    t["s"] = np.array([2.0], np_dt)
    t["m"] = rng.uniform(-2, 2, (mid,)).astype(np_dt)
    return t


# one element, around a vector, around a block's chunk, several chunks and a tail
@pytest.mark.parametrize("dt", ["f32", "f64"])
@pytest.mark.parametrize("shape,mid,inner", [((1, 1), 1, 1), ((3, 1), 1, 1), ((5, 1), 1, 1), ((1, 2047), 2047, 1), ((2, 1024), 1024, 1),
                                             ((7, 1171), 1171, 1), ((3, 5, 137), 5, 137), ((2, 260, 8), 260, 8)])
def test_run_stores_the_bits_of_its_commands(ctx, shape, mid, inner, dt):
    np_dt, code = (np.float32, _ffi.F32) if dt == "f32" else (np.float64, _ffi.F64)
    n = int(np.prod(shape))
    rng = np.random.default_rng(n + mid)

    def make(p):
        return [D.cmd_bin("mul", "vv", p["a"], p["b"], n, dtype=code, dst=p["c"]),
                D.cmd_bcast("add", p["c"], p["c"], p["m"], n // (mid * inner), mid, inner, dtype=code),
                D.cmd_unary("sigmoid", p["c"], n, dtype=code),
                D.cmd_unary("tanh", p["c"], n, dtype=code, dst=p["d"]),
                D.cmd_bin("pow", "vs", p["c"], p["s"], n, dtype=code, dst=p["a"]),
                D.cmd_bcast("sub", p["b"], p["d"], p["m"], n // (mid * inner), mid, inner, small_left=True, dtype=code)]
    _same(_both(ctx, make, _tensors(rng, shape, mid, np_dt)))


@pytest.mark.parametrize("dt", ["f32", "f64"])
def test_every_function_in_a_run(ctx, dt):
    np_dt, code = (np.float32, _ffi.F32) if dt == "f32" else (np.float64, _ffi.F64)
    n = 1031
    rng = np.random.default_rng(3)
    for u, b in zip(UNARY, (BINARY * 2)[:len(UNARY)]):
        def make(p):
            return [D.cmd_unary(u, p["a"], n, dtype=code, dst=p["c"]), D.cmd_bin(b, "vv", p["c"], p["b"], n, dtype=code, dst=p["d"]),
                    D.cmd_bin(b, "sv", p["s"], p["d"], n, dtype=code), D.cmd_leaky_relu(p["d"], p["a"], n, 0.1, dtype=code),
                    D.cmd_relu_bwd(p["b"], p["a"], p["a"], n, dtype=code), D.cmd_relu(p["a"], p["b"], n, dtype=code)]
        _same(_both(ctx, make, _tensors(rng, (n,), 1, np_dt)))


@pytest.mark.parametrize("seed", range(24))
def test_random_runs(ctx, seed):
    """Operands picked at random: values overwritten before, while and after others read them, more live values
    than the kernel keeps, runs longer than one launch takes, scalars that are elements of written tensors."""
    rng = np.random.default_rng(seed)
    np_dt, code, item = ((np.float32, _ffi.F32, 4), (np.float64, _ffi.F64, 8))[seed % 2]
    n = int(rng.integers(1, 5000))
    tensors = _tensors(rng, (n,), n, np_dt)

    def make(p):
        r = np.random.default_rng(seed + 1000)
        cmds = []
        for _ in range(int(r.integers(2, 20))):
            x, y, z = (p[k] for k in r.choice(list("abcd"), 3))
            kind = r.integers(5)
            fn = str(r.choice(["add", "sub", "mul", "lt", "gte"]))
            if kind == 0:
                cmds.append(D.cmd_bin(fn, "vv", x, y, n, dtype=code, dst=z))
            elif kind == 1:
                cmds.append(D.cmd_bin(fn, "vs", x, p["s"], n, dtype=code, dst=z))
            elif kind == 2:
                cmds.append(D.cmd_unary(str(r.choice(["tanh", "neg", "abs", "sigmoid"])), x, n, dtype=code, dst=z))
            elif kind == 3:
                cmds.append(D.cmd_bcast(fn, z, x, p["m"], 1, n, 1, small_left=bool(r.integers(2)), dtype=code))
            elif x != z:   # the scalar is an element of another tensor, which the run may have written
                cmds.append(D.cmd_bin(fn, "vs", z, x + item * int(r.integers(n)), n, dtype=code))
        return cmds
    _same(_both(ctx, make, tensors))


# the last size whose threads take one element each, the first of one vector each, tails of a vector; float64 past 16 MiB
@pytest.mark.parametrize("dt,mid,rows", [("f32", 640, 512), ("f32", 641, 512), ("f32", 327683, 1), ("f64", 640, 512), ("f64", 327681, 1),
                                         ("f64", 1048577, 2), ("f64", 2097153, 1)])
def test_runs_around_a_threads_share(ctx, dt, mid, rows):
    np_dt, code = (np.float32, _ffi.F32) if dt == "f32" else (np.float64, _ffi.F64)
    n = rows * mid
    heavy = ["exp", "softplus", "ln", "tanh"]

    def make(p):
        return [D.cmd_bin("mul", "vv", p["a"], p["b"], n, dtype=code, dst=p["c"]),
                D.cmd_bcast("add", p["c"], p["c"], p["m"], rows, mid, 1, dtype=code),
                D.cmd_unary(heavy[rows % 4], p["c"], n, dtype=code),
                D.cmd_bin("pow", "vs", p["c"], p["s"], n, dtype=code, dst=p["a"]),
                D.cmd_bin("sub", "vv", p["a"], p["b"], n, dtype=code, dst=p["d"]),
                D.cmd_relu(p["d"], p["d"], n, dtype=code)]
    _same(_both(ctx, make, _tensors(np.random.default_rng(n), (rows, mid), mid, np_dt)))
