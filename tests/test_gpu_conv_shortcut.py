"""The end of a residual block in one launch: main 1x1 convolution + projection shortcut (a second 1x1 convolution, any stride) + ReLU +
the next layers' Quantize, and the form that writes the quantised values alone, against the oracle's separate layers, bit for bit.
Semantics: Convolution::forward_int8 (src/layer/convolution.cpp:383-508), Eltwise sum (src/layer/eltwise.cpp:95-118), ReLU
(src/layer/relu.cpp:30-45), Quantize (src/layer/quantize.cpp:48-111)."""
import ctypes as C

import numpy as np
import pytest

from tests import cases
from oracle import oracle
from ncnn_amd.hip import Activation, ConvDesc, ConvFusion, ConvShortcut, DeviceBuffer, check, lib

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module")
def rt():
    import ncnn_amd
    return ncnn_amd.Runtime(0)


def _desc(batch, c, h, w, outc, stride):
    return ConvDesc(w, h, c, batch, outc, 1, 1, 1, 1, stride, stride, 0, 0, 0, 0, 0.0, 1)


def _operands(rt, seed, batch, c, h, w, outc, stride, bias, act, act_params):
    x, wq, b, ws, ins, _ = cases.conv_case(seed, c, h, w, outc, (1, 1), 1, 2, bias, True, batch=batch)
    d = oracle.make_desc((c, h, w), outc, (1, 1), (1, 1), (stride, stride), (0, 0, 0, 0), 0.0, int(bias), 1, 2, act, act_params)
    want = np.stack([oracle.convolution_int8(d, x[i], wq, b, ws, ins[0], None) for i in range(batch)])
    desc, size = _desc(batch, c, h, w, outc, stride), C.c_size_t()
    check(lib().ncnnhip_conv_nhwc_sizes(C.byref(desc), None, C.byref(size), None))
    packed = np.empty(size.value, np.int8)
    check(lib().ncnnhip_conv_pack_weights(C.byref(desc), np.ascontiguousarray(wq, np.int8).ctypes.data, packed.ctypes.data))
    keep = (rt.to_channels_last(x), rt.up(packed), rt.up(rt.fold_input_scales(ws, ins, outc)), rt.up(np.asarray(b, F)) if bias else None)
    return desc, keep, want


SHAPES = [
    # batch, main channels, h, w, output channels, shortcut channels, stride
    (1, 64, 5, 7, 40, 128, 1),  # 16 x 16 tiles, a channel tail and padding
    (1, 512, 7, 7, 2048, 1024, 2),  # 16 x 32
    (1, 256, 14, 14, 1024, 512, 2),  # 32 x 32
    (1, 64, 28, 28, 250, 1024, 2),  # 32 x 32, most of K in the shortcut
    (1, 64, 56, 55, 64, 64, 1),  # 32 x 32, a step of each
    (2, 1600, 6, 5, 24, 64, 3),  # one step of shortcut, two rounds of the main convolution
    (1, 64, 7, 7, 500, 5440, 1), (1, 5440, 7, 7, 500, 128, 2),  # 16 x 16, a K that goes on alone for rounds
    (1, 192, 7, 7, 2000, 6400, 1), (1, 4160, 7, 7, 2048, 1088, 1),  # 16 x 32, the same
    (1, 128, 28, 28, 256, 1600, 1), (1, 2560, 28, 28, 250, 192, 1),  # 32 x 32
    (1, 64, 56, 56, 256, 64, 1),  # the ring: 64-channel tiles
    (3, 128, 29, 27, 200, 192, 2),  # ragged pixels and channels
    (2, 64, 224, 224, 300, 64, 1),  # 128-channel tiles, the last mostly padding
]


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_projection_shortcut_in_the_sum(rt, shape):
    batch, c, h, w, outc, sc, stride = shape
    print("[case] conv shortcut", shape, flush=True)
    act, sact = ((3, (-0.5, 0.75)), (0, (0.0, 0.0))) if c == 128 else ((0, (0.0, 0.0)), (2, (0.1, 0.0))) if c == 256 else ((0, (0.0, 0.0)), (0, (0.0, 0.0)))
    desc, (x, wp, si, b), main = _operands(rt, c + outc, batch, c, h, w, outc, 1, True, *act)
    sdesc, (sx, swp, ssi, sb), side = _operands(rt, sc + outc + 1, batch, sc, h * stride - (stride > 1), w * stride - (stride > 1), outc, stride, c != 64, *sact)
    supported = C.c_int()
    check(lib().ncnnhip_conv_shortcut_supported(C.byref(desc), C.byref(sdesc), C.byref(supported)))
    assert supported.value == 1
    want = np.maximum((main + side).astype(F), 0)
    scale = F(100) / np.abs(want).max()
    want_q = oracle.quantize(want.reshape(batch * outc, -1), [scale]).reshape(want.shape)
    ocp = (outc + 15) // 16 * 16
    out, q8 = DeviceBuffer.empty((batch, h * w, ocp), F), DeviceBuffer.empty((batch, h * w, ocp), np.int8)
    short = ConvShortcut(C.pointer(sdesc), sx.ptr, swp.ptr, ssi.ptr, None if sb is None else sb.ptr, Activation.make(*sact))
    for with_out in (True, False):
        fu = ConvFusion(None, 1, q8.ptr, float(scale))
        check(lib().ncnnhip_conv_int8_nhwc_tail(C.byref(desc), x.ptr, wp.ptr, si.ptr, b.ptr, Activation.make(*act), C.byref(short), out.ptr if with_out else None,
                                                C.byref(fu), None, 0, rt.stream))
        raw = q8.to_numpy(rt.stream)
        assert not raw[:, :, outc:].any()
        assert np.array_equal(rt.from_channels_last(q8, batch, outc, h, w), want_q), with_out
        if with_out:
            assert np.array_equal(rt.from_channels_last(out, batch, outc, h, w), want)


@pytest.mark.parametrize("batch,c,hw,outc,kernel", [(1, 64, 5, 40, 1), (1, 64, 56, 64, 3), (16, 64, 56, 100, 1), (16, 64, 56, 64, 3), (12, 512, 7, 512, 3)])
def test_quantised_output_alone(rt, batch, c, hw, outc, kernel):
    """A residual blob, and no fp32 output, on each kernel that can be asked for it (few tiles, the ring, K split over workgroups)."""
    print("[case] conv quantised output alone", batch, c, hw, outc, kernel, flush=True)
    x, wq, b, ws, ins, _ = cases.conv_case(c + outc, c, hw, hw, outc, (kernel, kernel), 1, 2, True, True, batch=batch)
    p = kernel // 2
    d = oracle.make_desc((c, hw, hw), outc, (kernel, kernel), (1, 1), (1, 1), (p, p, p, p), 0.0, 1, 1, 2, 0, (0.0, 0.0))
    main = np.stack([oracle.convolution_int8(d, x[i], wq, b, ws, ins[0], None) for i in range(batch)])
    res = np.random.default_rng(outc).normal(0, 1, main.shape).astype(F)
    want = np.maximum((main + res).astype(F), 0)
    scale = F(100) / np.abs(want).max()
    want_q = oracle.quantize(want.reshape(batch * outc, -1), [scale]).reshape(want.shape)
    desc = ConvDesc(hw, hw, c, batch, outc, kernel, kernel, 1, 1, 1, 1, p, p, p, p, 0.0, 1)
    size, wsb = C.c_size_t(), C.c_size_t()
    check(lib().ncnnhip_conv_nhwc_sizes(C.byref(desc), None, C.byref(size), C.byref(wsb)))
    packed = np.empty(size.value, np.int8)
    check(lib().ncnnhip_conv_pack_weights(C.byref(desc), np.ascontiguousarray(wq, np.int8).ctypes.data, packed.ctypes.data))
    keep = (rt.to_channels_last(x), rt.up(packed), rt.up(rt.fold_input_scales(ws, ins, outc)), rt.up(np.asarray(b, F)), rt.to_channels_last(res))
    ws_dev = DeviceBuffer.zeros(max(wsb.value, 4), rt.stream)
    q8 = DeviceBuffer.empty((batch, hw * hw, (outc + 15) // 16 * 16), np.int8)
    fu = ConvFusion(keep[4].ptr, 1, q8.ptr, float(scale))
    check(lib().ncnnhip_conv_int8_nhwc_tail(C.byref(desc), keep[0].ptr, keep[1].ptr, keep[2].ptr, keep[3].ptr, Activation.make(0, (0.0, 0.0)), None, None, C.byref(fu),
                                            ws_dev.ptr, wsb.value, rt.stream))
    assert np.array_equal(rt.from_channels_last(q8, batch, outc, hw, hw), want_q)


def test_projection_shortcut_of_a_million_pixels(rt):
    """From 2^20 pixels on the ring finds the shortcut's pixel by whole divisions: images, rows and columns of a stride of 2."""
    batch, hw, c, outc = 3, 592, 64, 16
    print("[case] conv shortcut, a million pixels", flush=True)
    assert batch * hw * hw >= 1 << 20
    rng = np.random.default_rng(20)
    x, sx = (rng.integers(-127, 128, (batch, n, n, c), dtype=np.int8) for n in (hw, 2 * hw - 1))
    scales = rng.uniform(2000, 4000, (2, outc)).astype(F)
    bias = rng.uniform(-1, 1, outc).astype(F)
    sides, weights = [], []
    for blob, ws, b in ((x, scales[0], bias), (sx[:, ::2, ::2], scales[1], np.zeros(outc, F))):
        wq = rng.integers(-127, 128, (outc, c, 1, 1)).astype(np.int8)
        d = oracle.make_desc((c, hw, hw), outc, (1, 1), (1, 1), (1, 1), (0, 0, 0, 0), 0.0, 1, 1, 2, 0, (0.0, 0.0))
        sides.append(np.stack([oracle.convolution_int8(d, blob[i].transpose(2, 0, 1).astype(F), wq, b, ws, F(1), None) for i in range(batch)]))
        weights.append(wq)
    want = np.maximum((sides[0] + sides[1]).astype(F), 0)
    desc, sdesc = _desc(batch, c, hw, hw, outc, 1), _desc(batch, c, 2 * hw - 1, 2 * hw - 1, outc, 2)
    dev = [rt.up(v) for v in (x, sx)]
    packed = []
    for d, wq in zip((desc, sdesc), weights):
        p = np.empty(outc * c, np.int8)
        check(lib().ncnnhip_conv_pack_weights(C.byref(d), wq.ctypes.data, p.ctypes.data))
        packed.append(rt.up(p))
    folded = [rt.up(rt.fold_input_scales(ws, np.array([1], F), outc)) for ws in scales]
    b = rt.up(bias)
    out = DeviceBuffer.empty((batch, hw * hw, outc), F)
    act = Activation.make(0, (0.0, 0.0))
    short = ConvShortcut(C.pointer(sdesc), dev[1].ptr, packed[1].ptr, folded[1].ptr, None, act)
    fu = ConvFusion(None, 1, None, 0.0)
    check(lib().ncnnhip_conv_int8_nhwc_tail(C.byref(desc), dev[0].ptr, packed[0].ptr, folded[0].ptr, b.ptr, act, C.byref(short), out.ptr, C.byref(fu), None, 0, rt.stream))
    assert np.array_equal(rt.from_channels_last(out, batch, outc, hw, hw), want)


def test_pairs_that_are_refused(rt):
    supported = C.c_int(1)
    main = _desc(1, 64, 8, 8, 64, 1)
    for other in (_desc(1, 64, 8, 8, 48, 1), _desc(2, 64, 8, 8, 64, 1), _desc(1, 96, 8, 8, 64, 1), _desc(1, 64, 20, 16, 64, 2),
                  ConvDesc(8, 8, 64, 1, 64, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 0.0, 1), ConvDesc(6, 6, 64, 1, 64, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 0.0, 1),
                  ConvDesc(8, 8, 64, 1, 64, 1, 1, 1, 1, 1, 1, 0, 0, 0, 0, 1.0, 1)):
        check(lib().ncnnhip_conv_shortcut_supported(C.byref(main), C.byref(other), C.byref(supported)))
        assert supported.value == 0
