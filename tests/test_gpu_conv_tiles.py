"""The tiles the pipelined channels-last convolution takes by shape (64 x 64, 64 x 128 and 128 x 128 pixels x channels), in every
addressing mode, on pixel counts that leave a ragged last tile: bit for bit against the oracle, after the dispatch has
named the tile.  Semantics: Convolution::forward_int8 (src/layer/convolution.cpp:383-508)."""
import numpy as np
import pytest

from tests import cases
from oracle import oracle

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.mark.parametrize("batch,c,h,w,outc,kernel,term,fused,tile,addressing", [
    (52, 1024, 21, 23, 256, (1, 1), 102, False, (128, 128), 1),
    (52, 1024, 21, 23, 250, (1, 1), 2, False, (128, 128), 1),      # channel tail
    (52, 128, 21, 23, 256, (3, 3), 102, False, (128, 128), 3),
    (52, 112, 21, 23, 256, (3, 3), 2, False, (128, 128), 0),       # taps that are no whole steps
    (41, 512, 21, 23, 512, (1, 1), 2, False, (64, 128), 1),        # 8 steps on more tiles of 128 x 128 than fill the chip twice
    (41, 64, 21, 23, 256, (1, 1), 102, False, (64, 64), 1),        # one step
    (41, 512, 21, 23, 192, (1, 1), 102, False, (64, 64), 1),       # channels that no 128-wide tiles cover without more padding
    (41, 512, 21, 23, 512, (1, 1), 2, True, (64, 64), 1),
    (41, 512, 21, 23, 1024, (1, 1), 2, True, (64, 128), 1),
    (41, 64, 21, 23, 1024, (3, 3), 2, True, (64, 128), 3),         # 9 steps
    (52, 256, 21, 23, 250, (3, 3), 2, True, (128, 128), 3),        # a sum of 36 steps
    (50, 208, 15, 17, 512, (3, 3), 2, True, (128, 128), 0),        # 30, taps that are no whole steps
    (41, 128, 21, 23, 512, (3, 3), 2, True, (64, 128), 3),         # 18 steps on more than 512 tiles of 128 x 128
    (41, 160, 21, 23, 256, (3, 3), 2, False, (128, 128), 0),       # 23 steps on more than 300 of them
    (41, 128, 21, 23, 256, (3, 3), 102, False, (64, 128), 3),      # 18 on as many
], ids=str)
def test_tile_of_a_layer(batch, c, h, w, outc, kernel, term, fused, tile, addressing):
    import ncnn_amd
    pads = (kernel[0] // 2,) * 4
    route = cases.conv_route(batch, c, h, w, outc, kernel, pads=pads, act=0 if fused else 1, int8_out=term > 100, fused=fused)
    assert (route.kernel, route.tile_pixels, route.tile_channels, route.addressing, route.groups, route.splits) == (route.PIPELINED,) + tile + (addressing, 1, 1)
    x, wq, b, ws, ins, tops = cases.conv_case(21, c, h, w, outc, kernel, 1, term, True, True, batch=batch)
    d = oracle.make_desc((c, h, w), outc, kernel, (1, 1), (1, 1), pads, 0.0, 1, 1, term, 0 if fused else 1, (0.0, 0.0))
    checked = (0, 1, 20, 39, batch - 1)
    want = np.stack([oracle.convolution_int8(d, x[i], wq, b, ws, ins[0], None if tops is None else tops[0]) for i in checked])
    rt = ncnn_amd.Runtime(0)
    args = (x, wq, b, ws, ins, tops, outc, kernel, (1, 1), (1, 1), pads, 0.0, 1, term, 0 if fused else 1, (0.0, 0.0))
    if not fused:
        got = rt.conv_channels_last(*args)
        assert got.dtype == want.dtype and np.array_equal(got[list(checked)], want)
        return
    res = np.random.default_rng(22).normal(0, 1, (batch, outc, h, w)).astype(F)
    want = np.maximum((want + res[list(checked)]).astype(F), 0)
    scale = F(100) / np.abs(want).max()
    want_q = oracle.quantize(want.reshape(-1, w), [scale]).reshape(want.shape)
    got, got_q = rt.conv_channels_last(*args, residual=res, relu_after=True, quantise_scale=scale)
    assert np.array_equal(got[list(checked)], want)
    assert np.array_equal(got_q[list(checked)], want_q)
