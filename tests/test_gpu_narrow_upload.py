"""Planar fp32 images of at most 4 channels to 4 floats a pixel (ncnnhip_chw_to_nhwc4_f32), bit for bit: planes on 128-byte lines and off
them by any number of floats, at the edges of the kernels' pixel tiles, from device and page-locked memory; nothing beyond the blob is written."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hw", [1, 31, 33, 992, 993, 1023, 1024, 1025, 2049, 45232])
@pytest.mark.parametrize("c,batch", [(1, 3), (2, 1), (3, 2), (4, 2)])
def test_planes_on_and_off_lines(hw, c, batch):
    import torch
    import ncnn_amd
    from ncnn_amd.hip import check, lib
    stream = ncnn_amd.Runtime(0).stream
    for offset, pad, pinned in [(0, -hw % 32, False), (0, 0, True), (1, 0, False), (31, 1, False), (4, -hw % 4, True), (0, 17, False)]:
        print("[case] narrow upload", hw, c, batch, offset, pad, pinned, flush=True)
        cstep, nstep = hw + pad, (hw + pad) * c + (8 if pad else 0)
        host = torch.rand(offset + nstep * batch, generator=torch.Generator().manual_seed(hw + c))
        src = host.pin_memory() if pinned else host.cuda()
        got = torch.full((batch * hw * 4 + 64,), -7.0, device="cuda")
        torch.cuda.synchronize()
        check(lib().ncnnhip_chw_to_nhwc4_f32(C.c_void_p(src.data_ptr() + offset * 4), c, hw, batch, cstep, nstep, C.c_void_p(got.data_ptr()), stream))
        torch.cuda.synchronize()
        want = torch.zeros(batch, hw, 4)
        for n in range(batch):
            for q in range(c):
                at = offset + n * nstep + q * cstep
                want[n, :, q] = host[at:at + hw]
        assert torch.equal(got[:batch * hw * 4].cpu().view(batch, hw, 4), want) and bool((got[batch * hw * 4:] == -7.0).all())
