"""Which kernel and form a channels-last convolution takes: the dispatch's own answer (ncnnhip_conv_int8_nhwc_route), no GPU needed."""
import ctypes as C

import pytest

import cases

SAME3 = dict(pads=(1, 1, 1, 1))


@pytest.mark.parametrize("shape,options,kernel", [
    ((1, 512, 7, 7, 512, (3, 3)), SAME3, "FEW_TILES"),
    ((5, 512, 7, 8, 512, (3, 3)), SAME3, "PIPELINED"),
    ((1, 288, 12, 12, 160, (3, 3)), SAME3, "PIPELINED"),
    ((16, 64, 56, 56, 64, (3, 3)), SAME3, "RESIDENT"),
    ((32, 16, 112, 112, 96, (1, 1)), dict(int8_out=True), "POINTWISE"),
    ((32, 16, 112, 112, 96, (1, 1)), dict(int8_out=False), "PIPELINED"),
    ((2, 64, 45, 46, 64, (3, 3)), SAME3, "SMALL_TILE"),
    ((1, 256, 56, 56, 64, (1, 1)), dict(fused=True), "FEW_TILES"),
], ids=str)
def test_kernel_of_a_layer(shape, options, kernel):
    r = cases.conv_route(*shape, **options)
    assert r.kernel == getattr(r, kernel)


def test_forms_of_the_pipelined_kernel():
    r = cases.conv_route(5, 512, 7, 8, 512, (3, 3), **SAME3)
    assert (r.tile_pixels, r.tile_channels, r.addressing, r.groups, r.splits) == (64, 64, 3, 4, 3)
    r = cases.conv_route(1, 288, 12, 12, 160, (3, 3), **SAME3)  # K split over workgroups of one group
    assert (r.addressing, r.groups, r.splits) == (0, 1, 3)


@pytest.mark.parametrize("shape,options,tile", [
    ((128, 256, 14, 14, 256, (3, 3)), SAME3, (128, 128)), ((64, 256, 14, 14, 256, (3, 3)), SAME3, (64, 128)),
    ((128, 128, 28, 28, 128, (3, 3)), SAME3, (128, 128)),  # a long K of 128 channels and many pixels
    ((128, 128, 28, 28, 512, (1, 1)), dict(fused=True), (64, 128)), ((64, 128, 28, 28, 512, (1, 1)), dict(fused=True), (64, 64)),
    ((128, 512, 7, 7, 2048, (1, 1)), dict(fused=True), (64, 128)),
    # sums of a long K: by LDS, as other layers of that K
    ((64, 512, 14, 14, 512, (3, 3)), dict(fused=True, **SAME3), (128, 128)), ((80, 512, 14, 14, 1024, (3, 3)), dict(fused=True, **SAME3), (128, 128)),
    ((8, 256, 14, 14, 2048, (3, 3)), dict(fused=True, **SAME3), (64, 128)), ((64, 128, 14, 14, 1024, (3, 3)), dict(fused=True, **SAME3), (64, 128)),
    ((46, 512, 14, 14, 1024, (3, 3)), dict(fused=True, **SAME3), (64, 128)), ((48, 256, 14, 14, 1024, (3, 3)), SAME3, (64, 128)), ((56, 256, 14, 14, 1024, (3, 3)), SAME3, (128, 128)),
    ((32, 256, 14, 14, 256, (3, 3)), dict(fused=True, **SAME3), (64, 64)), ((32, 96, 14, 14, 1024, (3, 3)), dict(fused=True, **SAME3), (128, 128)),
    ((104, 128, 16, 16, 1024, (1, 1)), dict(fused=True), (64, 64)), ((112, 128, 16, 16, 1024, (1, 1)), dict(fused=True), (64, 128)),
    # to int8: strided, and one tile that is partly padding
    ((64, 64, 28, 28, 512, (1, 1)), dict(stride=(2, 2), int8_out=True), (64, 128)), ((64, 64, 28, 28, 512, (1, 1)), dict(stride=(2, 2)), (64, 64)),
    ((32, 64, 28, 28, 512, (1, 1)), dict(stride=(2, 2), int8_out=True), (64, 64)),
    ((16, 256, 56, 56, 96, (1, 1)), dict(int8_out=True), (64, 128)), ((16, 256, 56, 56, 128, (1, 1)), dict(int8_out=True), (64, 64)),
    ((32, 64, 28, 28, 384, (1, 1)), {}, (64, 64)), ((128, 320, 7, 7, 1280, (1, 1)), {}, (64, 128)),
    ((8, 32, 368, 368, 64, (1, 1)), {}, (128, 64)),
], ids=str)
def test_tile_of_the_pipelined_kernel(shape, options, tile):
    r = cases.conv_route(*shape, **options)
    assert (r.kernel, r.tile_pixels, r.tile_channels, r.groups, r.splits) == (r.PIPELINED,) + tile + (1, 1)


@pytest.mark.parametrize("threshold", [None, "40000", "1", "1000000"])
def test_pixel_threshold_of_the_resident_kernel(monkeypatch, threshold):
    """NCNNHIP_RESIDENT_MIN moves the threshold and nothing else: a long K on whole 128s of channels goes to the 128 x 128 tiles whether it is set or not."""
    monkeypatch.delenv("NCNNHIP_RESIDENT_MIN", raising=False)
    if threshold:
        monkeypatch.setenv("NCNNHIP_RESIDENT_MIN", threshold)
    r = cases.conv_route(64, 128, 28, 28, 128, (3, 3), **SAME3)
    assert (r.kernel, r.tile_pixels, r.tile_channels) == (r.PIPELINED, 128, 128)
    assert (cases.conv_route(16, 64, 56, 56, 64, (3, 3), **SAME3).kernel == r.RESIDENT) == (int(threshold or 40000) <= 16 * 56 * 56)
    assert (cases.conv_route(32, 128, 28, 28, 128, (3, 3), **SAME3).kernel == r.RESIDENT) == (threshold == "1")


@pytest.mark.parametrize("shape,tile", [((40, 128, 3000, 3000, 192, (1, 1)), (128, 64)), ((41, 128, 3700, 3700, 256, (1, 1)), (128, 128)), ((40, 128, 3001, 3000, 190, (2, 1)), (128, 64)),
                                        ((40, 128, 3701, 3700, 256, (2, 1)), (128, 128)), ((40, 112, 3001, 3000, 192, (2, 1)), (128, 64)), ((1, 128, 1500, 1500, 65536, (1, 1)), (128, 256)),
                                        ((1, 128, 1500, 1200, 32704, (1, 1)), (128, 64))], ids=str)
def test_outputs_of_more_tiles_than_a_launch_holds(shape, tile):
    """A launch counts its threads in 32 bits: outputs of 69 GB and more (137 GB in tiles of 64 x 128) take tiles that are large enough for that, and for the
    kernel's division of a tile's number by multiplication."""
    r = cases.conv_route(*shape, int8_out=True)
    pixels = shape[0] * (shape[2] - shape[5][0] + 1) * (shape[3] - shape[5][1] + 1)
    assert (r.kernel, r.tile_pixels, r.tile_channels) == (r.PIPELINED,) + tile
    tiles_m, tiles_n = -(-pixels // r.tile_pixels), -(-shape[4] // r.tile_channels)
    assert tiles_m * tiles_n * 256 < 1 << 32 and tiles_m * tiles_n * tiles_n < 1 << 32


def test_layers_that_are_refused():
    from ncnn_amd.hip import Activation, ConvDesc, ConvRoute, lib
    r, act = ConvRoute(), Activation.make(0, (0.0, 0.0))
    border = ConvDesc(8, 8, 64, 1, 64, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1.0, 1)
    assert lib().ncnnhip_conv_int8_nhwc_route(C.byref(border), act, 0, None, C.byref(r)) == 0 and r.kernel == r.GENERAL
    grouped = ConvDesc(8, 8, 64, 1, 64, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 0.0, 2)
    assert lib().ncnnhip_conv_int8_nhwc_route(C.byref(grouped), act, 0, None, C.byref(r)) != 0
    assert lib().ncnnhip_conv_int8_nhwc_route(None, act, 0, None, C.byref(r)) != 0


@pytest.mark.parametrize("hw,outc,tile,even,odd", [((4, 4), 64, (16, 16), 192, 641), ((14, 14), 256, (16, 16), 288, 401), ((7, 7), 496, (16, 16), 192, 641),
                                                   ((14, 14), 512, (16, 32), 80, 145), ((28, 28), 160, (16, 32), 80, 145), ((28, 28), 256, (32, 32), 48, 47)], ids=str)
def test_few_tiles_of_a_long_k_are_left_to_k_splits(hw, outc, tile, even, odd):
    for longest in (even, odd):
        r = cases.conv_route(1, 64 * longest, *hw, outc, (1, 1))
        assert (r.kernel, r.tile_pixels, r.tile_channels) == (r.FEW_TILES,) + tile
        r = cases.conv_route(1, 64 * (longest + 2), *hw, outc, (1, 1))
        assert r.kernel == r.PIPELINED and r.splits > 1


@pytest.mark.parametrize("batch,outc,int8_out,shortest", [(1, 256, True, 5), (1, 256, False, 3), (1, 512, True, 5), (1, 512, False, 3), (4, 256, True, 8), (4, 256, False, 6)])
def test_few_steps_of_a_strided_tap_are_left_to_the_ring(batch, outc, int8_out, shortest):
    for steps, kernel in ((shortest - 1, "PIPELINED"), (shortest, "FEW_TILES")):
        r = cases.conv_route(batch, 64 * steps, 28, 28, outc, (1, 1), stride=(2, 2), int8_out=int8_out)
        assert r.kernel == getattr(r, kernel)
    for kernel in ((1, 1), (3, 3)):  # dense, and several taps
        r = cases.conv_route(1, 64, 14, 14, outc, kernel, pads=(kernel[0] // 2,) * 4, int8_out=int8_out)
        assert r.kernel == r.FEW_TILES


def _pays(batch, hw, outc, c, shortcut_c, stride=2):
    from ncnn_amd.hip import ConvDesc, check, lib
    main = ConvDesc(hw, hw, c, batch, outc, 1, 1, 1, 1, 1, 1, 0, 0, 0, 0, 0.0, 1)
    side = ConvDesc(stride * hw, stride * hw, shortcut_c, batch, outc, 1, 1, 1, 1, stride, stride, 0, 0, 0, 0, 0.0, 1)
    r = C.c_int(-1)
    check(lib().ncnnhip_conv_shortcut_pays(C.byref(main), C.byref(side), C.byref(r)))
    return r.value


@pytest.mark.parametrize("batch,hw,outc,c,shortcut_c,pays", [
    # few tiles: both K together up to twice what one convolution may have there
    (1, 7, 512, 6400, 6400, 1), (1, 7, 2048, 5120, 5120, 1), (1, 7, 2048, 5120, 5184, 0), (1, 7, 2048, 5184, 5184, 1), (2, 14, 512, 3072, 3072, 1), (2, 14, 512, 4096, 4096, 0),
    (1, 28, 256, 64, 1024, 1),
    # 104 to 256 tiles of 64 x 64
    (1, 28, 512, 128, 256, 1), (4, 14, 1024, 256, 512, 1), (5, 14, 1024, 384, 768, 1), (1, 28, 512, 1024, 64, 0), (4, 7, 2048, 512, 1024, 0), (5, 14, 1024, 448, 768, 0),
    # more
    (16, 7, 2048, 512, 1024, 1), (6, 14, 1024, 640, 1280, 1), (6, 14, 1024, 640, 1344, 0), (16, 28, 512, 768, 1536, 1), (16, 28, 512, 832, 1536, 0),
    (64, 56, 256, 64, 64, 1), (64, 14, 1024, 512, 1024, 1), (64, 14, 1024, 576, 1024, 0),
    (1, 28, 512, 96, 256, 0),  # not a pair at all: channels that fill no whole step
], ids=str)
def test_shortcuts_that_pay(batch, hw, outc, c, shortcut_c, pays):
    assert _pays(batch, hw, outc, c, shortcut_c) == pays


def test_few_tiles_of_a_large_input():
    """Offsets of the kernel for few tiles are 32 bits wide: an input of 2 GiB goes to the ring, one of just below does not."""
    for batch, kernel in ((1, "FEW_TILES"), (2, "PIPELINED")):
        assert getattr((r := cases.conv_route(batch, 320, 1900, 1900, 64, (1, 1), stride=(190, 190))), kernel) == r.kernel
