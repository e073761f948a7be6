"""gh_elementwise_run: which elementwise commands of a submit become one pass.  Small tensors gain by every launch
saved; large ones only where a value is handed on, so commands that have nothing to do with each other stay apart."""
import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D

MIB = 1 << 20


def _run(cmds):
    lib = _ffi.load()
    return lib.gh_elementwise_run((_ffi.GhCmd * len(cmds))(*cmds), len(cmds))


def _tensors(count, n, item):
    """Addresses of tensors that lie apart."""
    room = (n * item + 255) // 256 * 256
    return [0x10000000 + i * room for i in range(count)]


@pytest.mark.parametrize("dtype,item", [(_ffi.F32, 4), (_ffi.F64, 8)])
def test_commands_that_share_nothing(dtype, item):
    for mib, least in ((1, 2), (16, 2), (32, 4), (64, 9)):   # MiB a tensor, commands from which on they go together
        n = mib * MIB // item
        p = _tensors(24, n, item)
        unary = [D.cmd_unary("neg", p[i], n, dtype=dtype, dst=p[8 + i]) for i in range(8)]
        binary = [D.cmd_bin("mul", "vv", p[i], p[8 + i], n, dtype=dtype, dst=p[16 + i]) for i in range(8)]
        bcast = [D.cmd_bcast("add", p[i], p[i], p[20], 1, n // 64, 64, dtype=dtype) for i in range(8)]
        reads = [D.cmd_unary("neg", p[0], n, dtype=dtype, dst=p[8]), D.cmd_unary("abs", p[0], n, dtype=dtype, dst=p[9])]
        for cmds in (unary, binary, bcast, reads):
            assert _run(cmds) == (len(cmds) if len(cmds) >= least else 1), (mib, cmds[0].opcode)


@pytest.mark.parametrize("dtype,item", [(_ffi.F32, 4), (_ffi.F64, 8)])
@pytest.mark.parametrize("mib", [1, 64, 256])
def test_values_handed_on(dtype, item, mib):
    n = mib * MIB // item
    x, y, z, t, p, q, two = _tensors(7, n, item)
    chain = [D.cmd_bin("mul", "vv", x, y, n, dtype=dtype, dst=z), D.cmd_bcast("add", z, z, q, n // 64, 64, 1, dtype=dtype),
             D.cmd_unary("sigmoid", z, n, dtype=dtype), D.cmd_unary("tanh", z, n, dtype=dtype, dst=t),
             D.cmd_bin("pow", "vs", z, two, n, dtype=dtype, dst=p)]
    assert _run(chain) == 5
    assert _run(chain[:1]) == 1
    # something unrelated between two that belong together: still a quarter of the passes less
    mixed = [chain[0], D.cmd_unary("neg", q, n, dtype=dtype, dst=t), chain[2]]
    assert _run(mixed) == 3
    # overwritten in place: one read and one write of two each
    assert _run([D.cmd_unary("neg", x, n, dtype=dtype), D.cmd_unary("abs", x, n, dtype=dtype)]) == 2


def test_what_is_no_run():
    n = 4096
    x, y, z = _tensors(3, n, 4)
    neg = D.cmd_unary("neg", x, n, dst=y)
    assert _run([neg, D.cmd_unary("neg", y, n - 1, dst=z)]) == 1                     # another size
    assert _run([neg, D.cmd_unary("neg", y, n, dtype=_ffi.F64, dst=z)]) == 1         # another type
    assert _run([neg, D.cmd_unary("neg", y + 4, n, dst=z)]) == 1                     # no whole vectors
    assert _run([neg, D.cmd_softmax(y, z, 64, 64)]) == 1
    assert _ffi.load().gh_elementwise_run(None, 0) == 0


@pytest.mark.parametrize("dtype,item", [(_ffi.F32, 4), (_ffi.F64, 8)])
@pytest.mark.parametrize("mib", [0.01, 1, 4, 16, 64])
def test_long_functions(dtype, item, mib):
    """Functions of many instructions cost a run as much as the launch they save: two of them do not make one."""
    n = int(mib * MIB) // item
    x, y, z, t, two = _tensors(5, n, item)
    f32 = dtype == _ffi.F32

    def twice(fn, times=2):
        return [D.cmd_unary(fn, x, n, dtype=dtype, dst=z)] + [D.cmd_unary(fn, z, n, dtype=dtype)] * (times - 1)
    for fn in ("sin", "cos", "ln", "log2", "log1p"):
        assert _run(twice(fn)) == (1 if f32 else 2), fn
    for fn in ("exp", "expm1"):
        assert _run(twice(fn)) == (1 if f32 and mib >= 4 else 2), fn
    assert _run(twice("softplus")) == (1 if mib < (16 if f32 else 4) else 2)
    for fn in ("neg", "sqrt", "inverse", "sigmoid", "tanh"):
        assert _run(twice(fn)) == 2, fn
    assert _run(twice("sin", 3)) == 3 and _run(twice("exp", 3)) == 3
    for fn in ("sin", "exp", "softplus", "log1p"):   # with one of few instructions all of them do
        assert _run([D.cmd_unary("abs", x, n, dtype=dtype, dst=z), D.cmd_unary(fn, z, n, dtype=dtype)]) == 2, fn
    mul, add = D.cmd_bin("mul", "vv", x, y, n, dtype=dtype, dst=z), D.cmd_bin("add", "vv", z, y, n, dtype=dtype)
    power, square = D.cmd_bin("pow", "vv", z, y, n, dtype=dtype), D.cmd_bin("pow", "vs", z, two, n, dtype=dtype)
    assert _run([mul, power]) == (1 if f32 and mib < 16 else 2)
    assert _run([mul, add, power]) == 3
    assert _run([power, power]) == 1
    assert _run([mul, square]) == 2 and _run([square, square]) == 1
