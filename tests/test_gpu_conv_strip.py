"""k_conv3x3_strip, the first layer of three or four channels over large images: the bits of the wide-image kernel, which takes
the same shapes, under every epilogue; and both against float64 sums."""
import numpy as np
import pytest

from tests.test_gpu_conv_lanes import _forward, _run
from tests.util import assert_bits_equal, rel_frobenius

pytestmark = pytest.mark.gpu

# B, C, H, W, F, padH: whole blocks of 64 columns; a last block of one lane, of lanes that move left, of two columns; fewer
# columns than a block's; runs of two to six rows and a last run that is shorter; filters short of a tile and past one
CASES = [(8, 3, 128, 128, 16, 1), (3, 3, 130, 132, 16, 1), (2, 3, 206, 194, 16, 1), (8, 4, 100, 100, 20, 1), (16, 3, 150, 62, 16, 1), (8, 3, 202, 322, 16, 1),
         (1, 3, 416, 416, 16, 1), (4, 4, 130, 130, 40, 1)]


def _epilogues(F):
    rng = np.random.default_rng(3)
    bn = [rng.standard_normal(F), rng.uniform(0.5, 2, F), rng.standard_normal(F), rng.standard_normal(F)]
    bn = [v.astype(np.float32) for v in bn]
    return [{}, {"act": "relu"}, {"act": "relu", "pool2": True}, {"act": "leaky", "alpha": 0.1, "bn": bn, "pool2": True}, {"act": "leaky", "alpha": 0.1, "bn": bn},
            {"act": "leaky", "alpha": -0.5}]


@pytest.mark.parametrize("cfg", CASES)
def test_bits_of_the_wide_image_kernel(ctx, cfg, monkeypatch):
    for kw in _epilogues(cfg[4]):
        monkeypatch.delenv("GORGONIA_HIP_CONV_NO_STRIP", raising=False)
        x, w, got = _run(ctx, cfg, "f32", **dict(kw))
        monkeypatch.setenv("GORGONIA_HIP_CONV_NO_STRIP", "1")
        _, _, want = _run(ctx, cfg, "f32", **dict(kw))
        assert_bits_equal(got, want, str(kw))
        if not kw:
            assert rel_frobenius(got, _forward(x, w, 1)) <= 1e-6   # sums of 36 products at most
