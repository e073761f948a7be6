"""The float64 form of k_conv3x3_lanes with one filter tile by two groups: its edges in pixels, filters and channels against
sums over shifted images."""
import ctypes

import pytest

from gorgonia_amd import _ffi
from gorgonia_amd import device as D
from tests.test_gpu_conv_lanes import _forward, _run
from tests.util import rel_frobenius

pytestmark = pytest.mark.gpu

# B, C, H, W, F, padH: whole tiles; filters short of a tile and odd rows; no and two rows of padding; seventeen quads, so
# that one wavefront has one more; two quads, so that two wavefronts have none
CASES = [(20, 64, 7, 7, 128, 1), (12, 24, 21, 19, 35, 1), (22, 72, 9, 13, 64, 0), (9, 40, 17, 18, 33, 2), (20, 68, 7, 7, 128, 1), (50, 8, 14, 14, 64, 1)]


@pytest.mark.parametrize("cfg", CASES)
def test_against_the_sums(ctx, cfg):
    B, C, H, W, F, padH = cfg
    args = (0x10000, 0x20000, 0x30000, B, C, H, W, F, 3, 3, (padH, 1))
    assert ctx.lib.gh_runs_straight(ctypes.byref(D.cmd_conv2d(*args, dtype=_ffi.F64))) == 1
    x, w, got = _run(ctx, cfg, "f64")
    assert rel_frobenius(got, _forward(x, w, padH)) <= 1e-14   # sums of at most 9 x 72 products, rounded as a walk: sqrt(648) x 2^-53 = 2.8e-15, and the reference's own
