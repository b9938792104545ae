"""The convolution kernel for few output tiles (tiles of 16 x 16, 16 x 32 and 32 x 32 pixels x channels, K split over a workgroup's
wavefronts) against the oracle, bit for bit, at the edges of its tiles, of its K runs and of the rule that chooses it.
Semantics: Convolution::forward_int8 (src/layer/convolution.cpp:383-508) per sample, batch as src/net.cpp:654-700."""
import numpy as np
import pytest

from tests import cases
from oracle import oracle

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module")
def rt():
    import ncnn_amd
    return ncnn_amd.Runtime(0)


NONE, SAME3 = (0, 0, 0, 0), (1, 1, 1, 1)
SHAPES = [
    # batch, c, h, w, outc, kernel, dilation, stride, pads.  Tiles of 16 x 16:
    (1, 64, 1, 1, 16, (1, 1), (1, 1), (1, 1), NONE),  # one pixel, one step: three wavefronts have none
    (1, 16, 5, 3, 17, (1, 1), (1, 1), (1, 1), NONE),  # a quarter of a step, a channel tail of one
    (2, 144, 7, 7, 40, (1, 1), (1, 1), (1, 1), NONE),  # the third step partly beyond the pixel
    (1, 3200, 3, 3, 40, (1, 1), (1, 1), (1, 1), NONE),  # 50 steps: two rounds of twelve, the second one step
    (1, 256, 14, 14, 256, (3, 3), (1, 1), (1, 1), SAME3),
    (1, 512, 7, 7, 512, (3, 3), (1, 1), (1, 1), SAME3),  # 72 steps
    (3, 128, 9, 5, 33, (3, 3), (2, 2), (1, 1), (2, 2, 2, 2)),
    (2, 192, 11, 9, 24, (1, 3), (1, 1), (2, 1), (0, 0, 1, 1)),  # a tap of three steps, uneven strides
    (1, 64, 64, 64, 16, (1, 1), (1, 1), (1, 1), NONE),  # 256 tiles
    (1, 3072, 2, 5, 40, (2, 2), (1, 1), (1, 1), (0, 0, 0, 0)),  # 192 steps, the longest K
    (1, 12416, 3, 3, 40, (1, 1), (1, 1), (1, 1), NONE),  # 194: K split over workgroups
    # 16 x 32
    (1, 64, 64, 64, 17, (1, 1), (1, 1), (1, 1), NONE),
    (1, 128, 28, 28, 128, (3, 3), (1, 1), (1, 1), SAME3),
    (1, 1024, 14, 14, 512, (1, 1), (1, 1), (2, 2), NONE),
    (1, 512, 7, 7, 2000, (1, 1), (1, 1), (1, 1), NONE),
    (1, 2560, 8, 32, 290, (1, 2), (1, 1), (1, 1), NONE),  # 80 steps, the longest even K
    (1, 5184, 8, 32, 258, (1, 1), (1, 1), (1, 1), NONE),  # 81, odd
    (1, 5248, 8, 32, 258, (1, 1), (1, 1), (1, 1), NONE),  # 82: K split over workgroups
    (1, 128, 28, 28, 200, (1, 1), (1, 1), (2, 2), NONE),  # a strided tap of two steps: the pipelined kernel's
    (1, 192, 28, 28, 200, (1, 1), (1, 1), (2, 2), NONE),  # three: here to fp32, there to int8
    # 32 x 32, and what the other kernels keep: four steps and fewer to int8, more than 48 steps, 257 tiles
    (1, 96, 63, 64, 60, (1, 1), (1, 1), (1, 1), NONE),
    (1, 320, 63, 64, 60, (1, 1), (1, 1), (1, 1), NONE),
    (4, 256, 14, 14, 256, (3, 3), (1, 1), (1, 1), SAME3),
    (5, 512, 7, 8, 512, (3, 3), (1, 1), (1, 1), SAME3),
    (1, 320, 8, 1028, 30, (1, 1), (1, 1), (1, 1), NONE),
]


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_few_tiles_kernel_matches_oracle(rt, shape):
    batch, c, h, w, outc, kernel, dilation, stride, pads = shape
    print("[case] conv few tiles", shape, flush=True)
    for term, act, ap, bias in [(2, 1, (0.0, 0.0), True), (102, 3, (0.0, 6.0), False), (2, 2, (0.1, 0.0), False), (102, 0, (0.0, 0.0), True)]:
        x, wq, b, ws, ins, tops = cases.conv_case(c + outc + term, c, h, w, outc, kernel, 1, term, bias, True, batch=batch)
        d = oracle.make_desc((c, h, w), outc, kernel, dilation, stride, pads, 0.0, int(bias), 1, term, act, ap)
        want = np.stack([oracle.convolution_int8(d, x[i], wq, b, ws, ins[0], None if tops is None else tops[0]) for i in range(batch)])
        got = rt.conv_channels_last(x, wq, b if bias else None, ws, ins, tops, outc, kernel, dilation, stride, pads, 0.0, 1, term, act, ap)
        assert got.dtype == want.dtype and np.array_equal(got, want), (term, act)


@pytest.mark.parametrize("c,h,w,outc", [(12416, 3, 3, 40), (5248, 8, 32, 258)])
def test_long_k_without_a_workspace(rt, c, h, w, outc):
    """A K that is split over workgroups given one, and taken by this kernel without."""
    import ctypes as C

    from ncnn_amd.hip import Activation, ConvDesc, DeviceBuffer, check, lib
    print("[case] conv few tiles, no workspace", c, h, w, outc, flush=True)
    assert cases.conv_route(1, c, h, w, outc, (1, 1)).splits > 1
    x, wq, b, ws, ins, _ = cases.conv_case(c, c, h, w, outc, (1, 1), 1, 2, True, True)
    d = oracle.make_desc((c, h, w), outc, (1, 1), (1, 1), (1, 1), NONE, 0.0, 1, 1, 2, 0, (0.0, 0.0))
    want = oracle.convolution_int8(d, x[0], wq, b, ws, ins[0], None)
    desc, size = ConvDesc(w, h, c, 1, outc, 1, 1, 1, 1, 1, 1, 0, 0, 0, 0, 0.0, 1), C.c_size_t()
    check(lib().ncnnhip_conv_nhwc_sizes(C.byref(desc), None, C.byref(size), None))
    packed = np.empty(size.value, np.int8)
    check(lib().ncnnhip_conv_pack_weights(C.byref(desc), np.ascontiguousarray(wq, np.int8).ctypes.data, packed.ctypes.data))
    keep = rt.to_channels_last(x), rt.up(packed), rt.up(rt.fold_input_scales(ws, ins, outc)), rt.up(np.asarray(b, F))
    out = DeviceBuffer.empty((1, h * w, (outc + 15) // 16 * 16), F)
    check(lib().ncnnhip_conv_int8_nhwc(C.byref(desc), keep[0].ptr, keep[1].ptr, keep[2].ptr, keep[3].ptr, None, Activation.make(0, (0.0, 0.0)), out.ptr, 1, 0, 0, None, 0,
                                       rt.stream))
    assert np.array_equal(rt.from_channels_last(out, 1, outc, h, w)[0], want)


@pytest.mark.parametrize("batch,c,hw,outc,kernel,pads,relu", [(1, 64, 5, 40, (1, 1), NONE, True), (1, 256, 14, 200, (3, 3), SAME3, False),
                                                              (1, 128, 28, 140, (1, 1), NONE, True), (1, 128, 63, 60, (1, 1), NONE, False)])
def test_few_tiles_kernel_fused_tail(rt, batch, c, hw, outc, kernel, pads, relu):
    """Residual, ReLU layer and the quantised copy for the next convolution, on each tile; a NaN of the residual stays."""
    print("[case] conv few tiles, fused tail", c, hw, outc, kernel, relu, flush=True)
    x, wq, b, ws, ins, _ = cases.conv_case(c + outc, c, hw, hw, outc, kernel, 1, 2, True, True, batch=batch)
    d = oracle.make_desc((c, hw, hw), outc, kernel, (1, 1), (1, 1), pads, 0.0, 1, 1, 2, 0, (0.0, 0.0))
    conv = np.stack([oracle.convolution_int8(d, x[i], wq, b, ws, ins[0], None) for i in range(batch)])
    res = np.random.default_rng(c).normal(0, 1, conv.shape).astype(F)
    want = (conv + res).astype(F)
    if relu:
        want = np.maximum(want, 0)
    scale = F(127) / np.abs(want).max()
    res.reshape(-1)[-1] = np.nan
    want.reshape(-1)[-1] = np.nan
    want_q = oracle.quantize(want.reshape(batch * outc, -1), [scale]).reshape(want.shape)
    got, got_q = rt.conv_channels_last(x, wq, b, ws, ins, None, outc, kernel, (1, 1), (1, 1), pads, 0.0, 1, 2, 0, (0.0, 0.0), residual=res, relu_after=relu,
                                       quantise_scale=scale)
    assert np.array_equal(got, want, equal_nan=True) and np.array_equal(got_q, want_q)


# Steps of K a wavefront has in flight at once (1, 2, 4, 6, 9, 12; on 32 x 32 tiles up to 9), rounds of them and eight wavefronts for more than 48 steps: each
# side of every change, dense and with taps, on 16 x 16, 16 x 32 and 32 x 32 tiles; whole runs of steps left to no wavefront.
@pytest.mark.parametrize("steps", [1, 2, 4, 5, 8, 9, 13, 16, 17, 24, 25, 36, 37, 48, 49, 72, 73, 96, 97, 192])
def test_few_tiles_kernel_runs_of_steps(rt, steps):
    print("[case] conv few tiles, steps", steps, flush=True)
    nine = max(1, steps // 9)
    for tile, batch, c, hw, outc, kernel, pads in ((16, 16), 1, 64 * steps, (3, 5), 33, (1, 1), NONE), ((16, 32), 1, 64 * steps, (16, 16), 290, (1, 1), NONE), \
            ((16, 32), 1, 64 * steps, (31, 32), 96, (1, 1), NONE), ((32, 32), 1, 64 * steps, (63, 64), 60, (1, 1), NONE), ((16, 16), 1, 64 * nine, (5, 4), 20, (3, 3), SAME3), \
            ((16, 32), 1, 64 * nine, (15, 16), 300, (3, 3), SAME3), ((32, 32), 4, 64 * nine, (13, 14), 250, (3, 3), SAME3):
        if batch * c * outc * hw[0] * hw[1] * kernel[0] * kernel[1] > 1 << 30:
            continue
        total = c * kernel[0] * kernel[1] // 64
        for term in (102, 2):
            route = cases.conv_route(batch, c, *hw, outc, kernel, pads=pads, act=1, int8_out=term > 100)
            longest = {(16, 16): (192, 641), (16, 32): (80, 145), (32, 32): (48, 48)}[tile][total % 2]
            taken = total <= longest and (tile != (32, 32) or total >= (5 if term > 100 else 2))
            assert (route.kernel == route.FEW_TILES) == taken and (not taken or (route.tile_pixels, route.tile_channels) == tile), (tile, total, term)
            if tile != (32, 32) and term == 2:
                continue
            x, wq, b, ws, ins, tops = cases.conv_case(steps + outc, c, hw[0], hw[1], outc, kernel, 1, term, True, True, batch=batch)
            d = oracle.make_desc((c, hw[0], hw[1]), outc, kernel, (1, 1), (1, 1), pads, 0.0, 1, 1, term, 1, (0.0, 0.0))
            got = rt.conv_channels_last(x, wq, b, ws, ins, tops, outc, kernel, (1, 1), (1, 1), pads, 0.0, 1, term, 1, (0.0, 0.0))
            for i in range(batch):
                assert np.array_equal(got[i], oracle.convolution_int8(d, x[i], wq, b, ws, ins[0], None if tops is None else tops[0])), (tile, total, term, i)
