"""Planar fp32 images of at most 4 channels to 4 floats a pixel (ncnnhip_chw_to_nhwc4_f32 and its form for
page-locked memory, each from both kinds of memory), bit for bit: planes on 128-byte lines and off
them by any number of floats, at the edges of the kernels' pixel tiles, from device and page-locked memory; nothing beyond the blob is written."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module")
def rt():
    import ncnn_amd
    return ncnn_amd.Runtime(0)


@pytest.fixture(scope="module")
def pinned():
    from ncnn_amd.hip import check, lib
    p = C.c_void_p()
    check(lib().ncnnhip_host_malloc(C.byref(p), 2 << 20))
    yield p
    check(lib().ncnnhip_host_free(p))


@pytest.mark.parametrize("hw", [1, 31, 33, 992, 993, 1023, 1024, 1025, 2049, 45232])
@pytest.mark.parametrize("c,batch", [(1, 3), (2, 1), (3, 2), (4, 2)])
def test_planes_on_and_off_lines(rt, pinned, hw, c, batch):
    from ncnn_amd.hip import check, lib
    for offset, pad, locked in [(0, -hw % 32, False), (0, 0, True), (1, 0, False), (31, 1, False), (4, -hw % 4, True), (0, 17, False)]:
        print("[case] narrow upload", hw, c, batch, offset, pad, locked, flush=True)
        cstep, nstep = hw + pad, (hw + pad) * c + (8 if pad else 0)
        host = np.random.default_rng(hw + c).random(offset + nstep * batch, dtype=F)
        if locked:
            assert host.nbytes <= 2 << 20
            C.memmove(pinned, host.ctypes.data, host.nbytes)
            base = pinned.value
        else:
            src = rt.up(host)
            base = src.ptr.value
        outs = []
        for entry in (lib().ncnnhip_chw_to_nhwc4_f32, lib().ncnnhip_chw_to_nhwc4_f32_from_host):
            got = rt.up(np.full(batch * hw * 4 + 64, -7, F))
            check(entry(C.c_void_p(base + offset * 4), c, hw, batch, cstep, nstep, got.ptr, rt.stream))
            outs.append(got.to_numpy(rt.stream))
        want = np.zeros((batch, hw, 4), F)
        for n in range(batch):
            for q in range(c):
                at = offset + n * nstep + q * cstep
                want[n, :, q] = host[at:at + hw]
        for out in outs:
            assert np.array_equal(out[:batch * hw * 4].reshape(batch, hw, 4), want) and (out[batch * hw * 4:] == -7).all()
