"""Which float32 products take their operands straight from memory and which are staged through LDS tiles, at shapes
where either was measured to be the slower by a tenth and more."""
import ctypes as C

import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D


def _straight(m, n, k, ta=False, tb=False, batch=1):
    cmd = D.cmd_gemm(0x10000, 0x20000, 0x30000, m, n, k, trans_a=ta, trans_b=tb, batch=batch, stride_a=m * k, stride_b=k * n, stride_c=m * n)
    return _ffi.load().gh_gemm_straight(C.byref(cmd))


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
    assert _ffi.load().gh_gemm_straight(C.byref(D.cmd_relu(0x1000, 0x2000, 16))) == 0


@pytest.mark.parametrize("m,n,k,ta,tb,slices", [(36, 907, 2696, False, False, 1), (300, 160, 4580, False, False, 1), (199, 280, 2287, True, False, 1),
                                                (116, 402, 13586, False, False, 1), (60, 560, 2300, False, False, 1), (48, 836, 2648, False, True, 1),
                                                (51, 641, 12494, False, False, 3), (424, 77, 20171, False, True, 3), (61, 451, 2913, False, True, 4),
                                                (343, 73, 5249, False, True, 3), (44, 612, 2104, True, False, 1),
                                                (324, 4, 2408, False, False, 4), (537, 1, 2784, True, False, 5), (12, 1336, 2496, False, False, 4), (12, 12, 7808, False, False, 15)])
def test_small_outputs_are_cut_where_slices_fill_an_idle_device(m, n, k, ta, tb, slices):
    assert _slices(m, n, k, ta, tb) == slices
