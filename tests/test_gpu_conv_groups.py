"""The pipelined convolution kernel with sixteen wavefronts per workgroup (K shared between four groups of four, int8
blobs with 64 x 64 tiles and at least 8 K steps) against the oracle: Convolution::forward_int8
(src/layer/convolution.cpp:383-508), every output bit for bit."""
import os

import numpy as np
import pytest

import cases
from oracle import oracle

pytestmark = pytest.mark.gpu
F = np.float32

# Beyond what the kernel for few tiles takes: more than 256 tiles of 32 x 32, or more than 48 steps and 256 tiles of 16 x 32 (pixels x channels),
# or steps that meet several taps.  The last two: addressing mode and K splits that the dispatch has to answer.
SHAPES = [
    # name, batch, c, h, w, outc, kernel, dilation, stride, pads, addressing, splits
    ("8 steps, two a group, 65 tiles", 1, 512, 5, 821, 64, (1, 1), (1, 1), (1, 1), (0, 0, 0, 0), 1, 1),
    ("9 steps: the last group has none, pixel and channel tails", 1, 576, 31, 89, 96, (1, 1), (1, 1), (1, 1), (0, 0, 0, 0), 1, 1),
    ("13 steps (the last half empty), 61 pixels in the last tile, 20 channels out", 1, 816, 63, 131, 20, (1, 1), (1, 1), (1, 1), (0, 0, 0, 0), 1, 1),
    ("1x1 stride 2, 16 steps, batch 3", 3, 1024, 47, 45, 136, (1, 1), (1, 1), (2, 2), (0, 0, 0, 0), 3, 1),
    ("3x3, 9 steps, batch 2", 2, 64, 45, 46, 64, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 3, 1),
    ("5x3 of 48 channels (a step meets several taps, K rounded up to 12 steps)", 1, 48, 10, 12, 72, (5, 3), (1, 1), (1, 1), (2, 2, 1, 1), 0, 1),
    ("3x3 dilated, 18 steps", 1, 128, 46, 45, 128, (3, 3), (2, 2), (1, 1), (2, 2, 2, 2), 3, 1),
    ("3x3, 36 steps, 76 tiles: one split", 6, 256, 14, 14, 256, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 3, 1),
    ("3x3, 72 steps, 40 tiles: three splits", 5, 512, 7, 8, 512, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 3, 3),
    ("1x1, 50 steps, 33 tiles: two splits of uneven groups", 1, 3200, 46, 45, 64, (1, 1), (1, 1), (1, 1), (0, 0, 0, 0), 1, 2),
    ("3x3 of 288 channels, 41 steps, 28 tiles: two splits, 21 steps and 20", 1, 288, 14, 14, 448, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 0, 2),
    ("1x1, 49 steps, 39 tiles: two splits, 25 steps and 24, two channels in the last tile", 1, 3136, 19, 43, 130, (1, 1), (1, 1), (1, 1), (0, 0, 0, 0), 1, 2),
]


@pytest.fixture(scope="module")
def rt():
    import ncnn_amd
    saved = os.environ.get("NCNNHIP_PATCH")
    os.environ["NCNNHIP_PATCH"] = "0"  # the small-tile kernel would take some of these
    yield ncnn_amd.Runtime(0)
    if saved is None:
        os.environ.pop("NCNNHIP_PATCH")
    else:
        os.environ["NCNNHIP_PATCH"] = saved


@pytest.mark.parametrize("shape", SHAPES, ids=[s[0] for s in SHAPES])
def test_sixteen_wavefronts_match_oracle(rt, shape):
    name, batch, c, h, w, outc, kernel, dilation, stride, pads, addressing, splits = shape
    print("[case] conv groups", name, flush=True)
    rng = np.random.default_rng(len(name))
    for term, act, ap in [(1, 1, (0.0, 0.0)), (102, 3, (0.0, 6.0)), (2, 2, (0.1, 0.0)), (101, 0, (0.0, 0.0))]:
        x, wq, b, ws, ins, tops = cases.conv_case(len(name) + term, c, h, w, outc, kernel, 1, term, True, True, batch=batch)
        d = oracle.make_desc((c, h, w), outc, kernel, dilation, stride, pads, 0.0, 1, 1, term, act, ap)
        route = cases.conv_route(batch, c, h, w, outc, kernel, dilation, stride, pads, act, ap, term > 100, term == 2)
        assert (route.kernel, route.groups, route.addressing, route.splits) == (route.PIPELINED, 4, addressing, splits)
        want = np.stack([oracle.convolution_int8(d, x[i], wq, b, ws, ins[0], None if tops is None else tops[0]) for i in range(batch)])
        got = rt.conv_channels_last(x, wq, b, ws, ins, tops, outc, kernel, dilation, stride, pads, 0.0, 1, term, act, ap)
        assert got.dtype == want.dtype and np.array_equal(got, want), (term, act)
        if term == 2:  # the fused tail: residual, ReLU, quantised copy
            res = rng.uniform(-2, 2, want.shape).astype(F)
            got, q8 = rt.conv_channels_last(x, wq, b, ws, ins, tops, outc, kernel, dilation, stride, pads, 0.0, 1, term, act, ap,
                                            residual=res, relu_after=True, quantise_scale=F(30.0))
            added = np.maximum(want + res, F(0))
            assert np.array_equal(got, added)
            assert np.array_equal(q8, oracle.quantize(added.reshape(-1, added.shape[-1]), [F(30.0)]).reshape(added.shape))
