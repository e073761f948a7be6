"""Which 3x3 filter gradients walk rows straight from memory and which are staged in tiles, at shapes where either was
measured to be the slower by a tenth and more."""
import ctypes as C

import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D


def _straight(cfg, dtype):
    B, Cn, H, W, F, pad = cfg
    cmd = D.cmd_conv2d_bwd_filter(0x10000, 0x20000, 0x30000, B, Cn, H, W, F, 3, 3, (pad, pad), dtype=dtype)
    return _ffi.load().gh_runs_straight(C.byref(cmd))


@pytest.mark.parametrize("cfg", [(12, 249, 20, 20, 376, 0), (2, 279, 53, 53, 237, 1), (46, 104, 69, 6, 500, 1), (28, 229, 14, 14, 168, 0),
                                 (32, 85, 37, 6, 295, 0), (22, 152, 17, 17, 125, 1), (12, 17, 62, 33, 165, 1), (3, 22, 10, 10, 228, 1)])
def test_float32_staged(cfg):
    assert _straight(cfg, _ffi.F32) == 0


@pytest.mark.parametrize("cfg", [(8, 16, 104, 104, 32, 1), (8, 32, 52, 52, 64, 1), (8, 64, 26, 26, 128, 1), (8, 128, 52, 52, 256, 1), (8, 3, 208, 208, 16, 1),
                                 (48, 347, 40, 40, 9, 1), (47, 159, 17, 48, 32, 1), (54, 14, 14, 197, 50, 0), (26, 8, 177, 177, 17, 0)])
def test_float32_straight(cfg):
    assert _straight(cfg, _ffi.F32) == 1


@pytest.mark.parametrize("cfg,straight", [((55, 21, 90, 3, 157, 1), 0), ((40, 130, 11, 11, 252, 1), 0), ((3, 26, 13, 13, 67, 1), 0),
                                          ((50, 32, 14, 14, 64, 1), 1), ((50, 64, 7, 7, 128, 1), 1), ((50, 1, 28, 28, 32, 1), 1),
                                          ((1, 9, 30, 30, 16, 1), 1), ((8, 278, 94, 94, 12, 1), 1)])
def test_float64(cfg, straight):
    assert _straight(cfg, _ffi.F64) == straight


def test_other_commands():
    lib = _ffi.load()
    assert lib.gh_runs_straight(C.byref(D.cmd_conv2d(0x10000, 0x20000, 0x30000, 1, 512, 13, 13, 1024, 3, 3, (1, 1)))) == 1
    assert lib.gh_runs_straight(C.byref(D.cmd_conv2d(0x10000, 0x20000, 0x30000, 128, 32, 14, 14, 64, 3, 3, (1, 1)))) == 0
    assert lib.gh_runs_straight(C.byref(D.cmd_conv2d_bwd_data(0x10000, 0x20000, 0x30000, 2, 64, 26, 26, 128, 3, 3, (1, 1)))) == 1
    assert lib.gh_runs_straight(C.byref(D.cmd_conv2d_bwd_data(0x10000, 0x20000, 0x30000, 2, 64, 26, 26, 128, 3, 3, (1, 1), (2, 2)))) == 0
    assert lib.gh_runs_straight(C.byref(D.cmd_conv2d(0x10000, 0x20000, 0x30000, 50, 32, 14, 14, 64, 3, 3, (1, 1), dtype=_ffi.F64))) == 1
    assert lib.gh_runs_straight(C.byref(D.cmd_conv2d_bwd_data(0x10000, 0x20000, 0x30000, 50, 32, 14, 14, 64, 3, 3, (1, 1), dtype=_ffi.F64))) == 1
    assert lib.gh_runs_straight(C.byref(D.cmd_relu(0x1000, 0x2000, 16))) == 0 and lib.gh_runs_straight(None) == 0
