"""Which products take their operands straight from memory and which are staged through LDS tiles, at shapes
where either was measured to be the slower by a tenth and more."""
import ctypes as C

import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D


def _straight(m, n, k, ta=False, tb=False, batch=1):
    cmd = D.cmd_gemm(0x10000, 0x20000, 0x30000, m, n, k, trans_a=ta, trans_b=tb, batch=batch, stride_a=m * k, stride_b=k * n, stride_c=m * n)
    return _ffi.load().gh_runs_straight(C.byref(cmd))


def _slices(m, n, k, ta=False, tb=False):
    sp = C.c_int(0)
    _ffi.load().gh_gemm_route(C.byref(D.cmd_gemm(0x10000, 0x20000, 0x30000, m, n, k, trans_a=ta, trans_b=tb)), C.byref(sp))
    return sp.value


@pytest.mark.parametrize("m,n,k,ta,tb", [(6, 103, 9561, True, False), (4, 347, 8609, True, False), (8, 60, 10257, False, True),
                                         (5, 81, 12018, True, False), (12, 6, 24972, False, True), (560, 9, 11892, True, True),
                                         (468, 24, 1430, True, True), (24, 1724, 5027, True, True), (9, 1481, 14476, True, False),
                                         (13, 5, 1392, False, True)])
def test_long_contractions_into_few_tiles_are_cut_among_workgroups(m, n, k, ta, tb):
    assert _straight(m, n, k, ta, tb) == 0 and _slices(m, n, k, ta, tb) > 8


@pytest.mark.parametrize("m,n,k,ta,tb", [(2471, 236, 723, True, True), (238, 1547, 20324, True, True), (181, 1838, 20758, True, True),
                                         (7, 221, 237, True, True), (346, 7, 322, True, True), (10, 65, 441, True, False),
                                         (73, 183, 400, True, True)])
def test_others_stay_with_their_workgroup(m, n, k, ta, tb):
    assert _straight(m, n, k, ta, tb) == 1


def test_slabs_fit_any_scratch():
    """More than the fixed scratch's 16 MiB of slabs: the kernel that needs none."""
    assert _slices(600, 850, 9000, True, True) * 600 * 850 * 4 <= 16 << 20 or _straight(600, 850, 9000, True, True) == 1
    assert _straight(64, 64, 64) == 0      # one small tile
    assert _straight(1, 300, 784) == 1     # one row
    assert _ffi.load().gh_runs_straight(C.byref(D.cmd_relu(0x1000, 0x2000, 16))) == 0


@pytest.mark.parametrize("m,n,k,ta,tb,slices", [(36, 907, 2696, False, False, 1), (300, 160, 4580, False, False, 1), (199, 280, 2287, True, False, 1),
                                                (116, 402, 13586, False, False, 1), (60, 560, 2300, False, False, 1), (48, 836, 2648, False, True, 1),
                                                (51, 641, 12494, False, False, 3), (424, 77, 20171, False, True, 3), (61, 451, 2913, False, True, 4),
                                                (343, 73, 5249, False, True, 3), (44, 612, 2104, True, False, 1),
                                                (324, 4, 2408, False, False, 4), (537, 1, 2784, True, False, 5), (12, 1336, 2496, False, False, 4), (12, 12, 7808, False, False, 15)])
def test_small_outputs_are_cut_where_slices_fill_an_idle_device(m, n, k, ta, tb, slices):
    assert _slices(m, n, k, ta, tb) == slices


@pytest.mark.parametrize("m,n,batch", [(1952, 1716, 1), (248, 164, 24), (4096, 4096, 1), (3060, 632, 1)])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True)])
@pytest.mark.parametrize("k", [4, 24, 96, 128])
def test_short_contractions_over_many_aligned_tiles_are_staged(m, n, batch, ta, tb, k):
    assert _straight(m, n, k, ta, tb, batch) == 0


@pytest.mark.parametrize("m,n,k,ta,tb,batch,straight", [
    (1954, 1715, 24, False, False, 1, 0), (1954, 1715, 64, False, False, 1, 1),      # rows that 16-byte loads cannot take
    (4001, 3001, 40, True, False, 1, 0), (505, 274, 48, True, False, 9, 1),
    (505, 274, 24, False, True, 9, 0), (500, 500, 8, False, True, 4, 0), (500, 500, 16, False, True, 4, 1),
    (2000, 8, 8, False, True, 4, 1), (128, 128, 12, False, False, 32, 1), (128, 128, 9, True, False, 32, 1),
    (200, 200, 24, True, True, 1, 0), (200, 200, 16, True, True, 1, 1), (200, 200, 48, True, True, 1, 1),
    (4, 3008, 8, True, True, 1, 0), (7, 194, 5, True, False, 1, 0),
    (1952, 1716, 256, True, False, 1, 0), (1952, 1716, 256, False, True, 1, 0), (249, 164, 256, False, True, 23, 1),
    (1952, 1716, 400, False, False, 1, 1), (1676, 2628, 192, False, False, 1, 1),
    (338, 182, 2, False, True, 64, 1), (230, 2495, 7, True, False, 24, 0), (1408, 260, 3, True, True, 8, 1), (4012, 7, 3, False, True, 8, 1), (24, 1260, 76, False, False, 24, 1),
    (12, 9, 27, False, True, 24, 1)])
def test_short_contractions(m, n, k, ta, tb, batch, straight):
    assert _straight(m, n, k, ta, tb, batch) == straight


@pytest.mark.parametrize("m,n,k,batch,straight", [
    (560, 1680, 12, 1, 0), (104, 936, 8, 24, 0), (1416, 3936, 16, 5, 0), (2000, 2000, 32, 1, 0), (2000, 2000, 48, 1, 0), (160, 499, 16, 16, 0),
    (255, 3906, 12, 8, 0), (300, 1868, 4, 1, 0),                                                     # staged
    (160, 499, 48, 16, 1), (128, 128, 5, 32, 1), (2000, 2000, 64, 1, 1), (1416, 3936, 64, 1, 1), (1543, 777, 24, 1, 1), (500, 500, 8, 1, 1), (300, 40, 12, 5, 1),
    (777, 1543, 1021, 1, 1),
    (64, 64, 64, 1, 0), (100, 100, 500, 1, 0)])                                # a tile a workgroup
def test_float64(m, n, k, batch, straight):
    cmd = D.cmd_gemm(0x10000, 0x20000, 0x30000, m, n, k, batch=batch, stride_a=m * k, stride_b=k * n, stride_c=m * n, dtype=_ffi.F64)
    assert _ffi.load().gh_runs_straight(C.byref(cmd)) == straight
