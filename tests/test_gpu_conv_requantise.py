"""Requantising epilogues that fold a ReLU, a clip or no activation into the clamp and round by one conversion, in the pipelined and the
pointwise convolution kernel, against the oracle bit for bit: sums on exact halves, clips with and without a negative bound, scales at
which a value may leave the 32-bit range (the form as written runs then), and an output scale that is negative.
Semantics: Convolution::forward_int8 (src/layer/convolution.cpp:370-512), src/layer/fused_activation.h:25-33."""
import numpy as np
import pytest

from tests import cases
from oracle import oracle

pytestmark = pytest.mark.gpu
F = np.float32
NONE, SAME3 = (0, 0, 0, 0), (1, 1, 1, 1)


@pytest.fixture(scope="module")
def rt():
    import ncnn_amd
    return ncnn_amd.Runtime(0)


# c, h, w, outc, kernel, pads: tiles of 64 x 64 with channel and pixel tails; 64 x 128; K over groups of wavefronts; the pointwise kernel (2^16 pixels)
SHAPES = [(48, 96, 97, 72, (1, 1), NONE), (64, 120, 121, 136, (1, 1), NONE), (96, 61, 67, 200, (3, 3), SAME3), (576, 48, 49, 90, (1, 1), NONE),
          (16, 256, 257, 36, (1, 1), NONE)]


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("act,ap", [(0, (0.0, 0.0)), (1, (0.0, 0.0)), (3, (0.0, 6.0)), (3, (0.5, 40.0)), (3, (-1.5, 30.0))], ids=str)
@pytest.mark.parametrize("top", [1.0, 1e12, -1.0])
def test_folded_requantisation_matches_oracle(rt, shape, act, ap, top):
    c, h, w, outc, kernel, pads = shape
    print("[case] conv requantise", shape, act, ap, top, flush=True)
    x, wq, b, _, _, _ = cases.conv_case(c + outc, c, h, w, outc, kernel, 1, 102, True, True)
    # powers of two: a sum of 2^-6 steps on both sides of zero, every half of the output's steps among the values
    x, ws, ins, tops = np.clip(x, -8, 8).astype(x.dtype), np.full(outc, 32, F), np.array([2], F), np.array([top], F)
    b = (np.round(b * 640) / 64).astype(F)
    d = oracle.make_desc((c, h, w), outc, kernel, (1, 1), (1, 1), pads, 0.0, 1, 1, 102, act, ap)
    want = oracle.convolution_int8(d, x[0], wq, b, ws, ins[0], tops[0])
    got = rt.conv_channels_last(x, wq, b, ws, ins, tops, outc, kernel, (1, 1), (1, 1), pads, 0.0, 1, 102, act, ap)[0]
    assert got.dtype == want.dtype and np.array_equal(got, want)
    if top == 1.0 and act < 3:
        assert len(np.unique(want)) > 60
