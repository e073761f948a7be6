"""Which float32 products run on the bf16 matrix instructions, at shapes where either way was measured to be the slower one."""
import ctypes as C

import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D


@pytest.mark.parametrize("m,n,k,ta,tb,batch,split", [
    (4096, 4096, 4096, False, False, 1, 1), (512, 512, 512, False, False, 64, 1), (2048, 2048, 2048, True, False, 1, 1), (1000, 1000, 1025, False, True, 1, 1),
    (500, 500, 500, False, False, 8, 1), (4096, 4096, 128, False, False, 1, 1), (2000, 2000, 47, False, False, 1, 1),
    (165, 2325, 1105, True, False, 1, 0), (300, 4000, 300, False, False, 1, 0), (1241, 199, 90, True, False, 1, 0),      # too few tiles, or a few us either way
    (4096, 4096, 15, False, False, 1, 0), (128, 1152, 625, False, False, 1, 0), (4096, 1, 4096, False, False, 1, 0)])
def test_products_on_the_bf16_instructions(m, n, k, ta, tb, batch, split):
    cmd = D.cmd_gemm(0x10000, 0x20000, 0x30000, m, n, k, trans_a=ta, trans_b=tb, batch=batch, stride_a=m * k, stride_b=k * n, stride_c=m * n)
    assert _ffi.load().gh_runs_split(C.byref(cmd)) == split
    cmd = D.cmd_gemm(0x10000, 0x20000, 0x30000, m, n, k, batch=batch, stride_a=m * k, stride_b=k * n, stride_c=m * n, dtype=_ffi.F64)
    assert _ffi.load().gh_runs_split(C.byref(cmd)) == 0
