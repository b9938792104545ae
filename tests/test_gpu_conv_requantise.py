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


# c, h, w, outc, kernel, pads, and what the dispatch has to answer (tile of channels, groups of wavefronts that share K, splits of K): tiles of 64 x 64
# with channel and pixel tails; 64 x 128; K over groups of wavefronts, dense and with taps; K split over workgroups of four groups and of one; the
# pointwise kernel (2^16 pixels)
SHAPES = [(48, 96, 97, 72, (1, 1), NONE, (64, 1, 1)), (64, 240, 241, 128, (1, 1), NONE, (128, 1, 1)), (96, 61, 67, 200, (3, 3), SAME3, (64, 4, 1)),
          (576, 60, 61, 90, (1, 1), NONE, (64, 4, 1)), (288, 14, 14, 448, (3, 3), SAME3, (64, 4, 2)), (288, 12, 12, 160, (3, 3), SAME3, (64, 1, 3)),
          (16, 256, 257, 36, (1, 1), NONE, None)]


def _takes_its_route(shape, act, ap):
    c, h, w, outc, kernel, pads, form = shape
    r = cases.conv_route(1, c, h, w, outc, kernel, pads=pads, act=act, act_params=ap, int8_out=True)
    assert r.kernel == r.POINTWISE if form is None else (r.kernel, r.tile_channels, r.groups, r.splits) == (r.PIPELINED,) + form


def _operands(shape):
    c, h, w, outc, kernel, pads, _ = shape
    x, wq, b, _, _, _ = cases.conv_case(c + outc, c, h, w, outc, kernel, 1, 102, True, True)
    # powers of two: a sum of 2^-6 steps on both sides of zero, every half of the output's steps among the values
    return np.clip(x, -8, 8).astype(x.dtype), wq, (np.round(b * 640) / 64).astype(F), np.full(outc, 32, F), np.array([2], F)


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("act,ap", [(0, (0.0, 0.0)), (1, (0.0, 0.0)), (3, (0.0, 6.0)), (3, (0.5, 40.0)), (3, (-1.5, 30.0))], ids=str)
@pytest.mark.parametrize("top", [1.0, 1e12, -1.0])
def test_folded_requantisation_matches_oracle(rt, shape, act, ap, top):
    c, h, w, outc, kernel, pads, _ = shape
    print("[case] conv requantise", shape, act, ap, top, flush=True)
    _takes_its_route(shape, act, ap)
    x, wq, b, ws, ins = _operands(shape)
    tops = np.array([top], F)
    d = oracle.make_desc((c, h, w), outc, kernel, (1, 1), (1, 1), pads, 0.0, 1, 1, 102, act, ap)
    want = oracle.convolution_int8(d, x[0], wq, b, ws, ins[0], tops[0])
    got = rt.conv_channels_last(x, wq, b, ws, ins, tops, outc, kernel, (1, 1), (1, 1), pads, 0.0, 1, 102, act, ap)[0]
    assert got.dtype == want.dtype and np.array_equal(got, want)
    if top == 1.0 and act < 3:
        assert len(np.unique(want)) > 60


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("act,ap", [(0, (0.0, 0.0)), (1, (0.0, 0.0)), (3, (0.0, 6.0))], ids=str)
@pytest.mark.parametrize("other", [1e12, -1.0])
def test_wavefronts_that_choose_different_epilogues(rt, shape, act, ap, other):
    """Output scales that let one block of 32 channels fold and the next one not: the wavefronts of one workgroup go different ways."""
    c, h, w, outc, kernel, pads, _ = shape
    print("[case] conv requantise, mixed", shape, act, ap, other, flush=True)
    x, wq, b, ws, ins = _operands(shape)
    folds = np.arange(outc) // 32 % 2 == 0
    d = oracle.make_desc((c, h, w), outc, kernel, (1, 1), (1, 1), pads, 0.0, 1, 1, 102, act, ap)
    want = np.where(folds[:, None, None], *[oracle.convolution_int8(d, x[0], wq, b, ws, ins[0], F(top)) for top in (1.0, other)])
    tops = np.where(folds, F(1), F(other)).astype(F)
    got = rt.conv_channels_last(x, wq, b, ws, ins, tops, outc, kernel, (1, 1), (1, 1), pads, 0.0, 1, 102, act, ap)[0]
    assert got.dtype == want.dtype and np.array_equal(got, want)
