"""The int8 Gemm on rows that begin and end at any byte, at the edges of its tiles, K steps and dispatch: against the oracle, bit for
bit (src/layer/gemm.cpp:745-966)."""
import ctypes as C

import numpy as np
import pytest

from ncnn_amd.hip import DeviceBuffer, check, lib
from oracle import oracle
from tests import cases, npref

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    import ncnn_amd
    return ncnn_amd.Runtime(0)


SHAPES = [
    # K: below a vector, one vector, around the few-row kernel's 64 and the tiles' 128 bytes, several steps with every kind of rest
    (65, 63, 15), (17, 64, 16), (63, 65, 17), (64, 129, 63), (129, 64, 65), (127, 128, 127), (128, 127, 128), (66, 70, 129), (130, 66, 143), (70, 70, 271), (64, 64, 400),
    # few rows (one workgroup per 16 rows of B), with K of 0 and more whole 64-byte steps
    (1, 64, 16), (3, 65, 63), (16, 79, 65), (17, 100, 321), (2, 63, 77), (1, 130, 2047),
    # long K on few tiles: eight wavefronts with runs of several K steps, the last cut
    (70, 65, 3072), (130, 65, 3073), (65, 66, 3200), (64, 64, 3327),
    # four wavefronts a tile of 32 x 32 from 257 tiles, some without a step; 64 x 64 tiles with eight from 641 tiles and K = 3072
    (300, 900, 144), (260, 1000, 1039), (16, 9000, 48), (620, 1000, 528), (768, 1024, 80), (530, 1000, 3088), (896, 768, 3088),
    # beyond the streaming kernel (450 tiles of 32 x 32, 640 or 1024 where rows are aligned): one and two groups of wavefronts per tile of 64 x 64
    (700, 700, 65), (720, 650, 271), (1000, 700, 528), (470, 970, 3073), (465, 990, 3327),
    # cut tiles of aligned rows leave the streaming kernel from 513 tiles and K = 2944 on: the last it keeps on either side, and the first it does not
    (500, 1000, 2944), (520, 1000, 2928), (513, 1000, 2944),
    # 257 to 512 tiles of 64 x 64 that are at most 256 of 96 x 64, in one and two groups of wavefronts; more of them, at most 256 of 96 x 96; and neither
    (1057, 1025, 273), (1056, 1024, 271), (1153, 961, 2992), (1100, 1000, 912), (1100, 1000, 3073), (1057, 1025, 3200), (2881, 705, 401), (1440, 1536, 1007), (1153, 1537, 655),
    (2305, 705, 401),
    # 128 x 128 tiles from 1536 tiles of 64 x 64
    (2497, 2497, 33), (1, 5000, 50), (3000, 2176, 130),
]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_gemm_int8_any_shape_equals_the_oracle(rt, m, n, k):
    print("[case]", m, n, k, flush=True)
    a, bq, sb, bias = cases.gemm_case(m + n + k, m, n, k, per_col=k % 2 == 0)
    aq, sa = rt.gemm_quantize_rows(a)
    want_q, want_s = oracle.gemm_quantize_rows(a)
    assert np.array_equal(aq, want_q) and np.array_equal(sa, want_s)
    want, wacc = oracle.gemm_int8(aq, bq, sa, sb, bias, 4, 0.5, 1.5, False, want_acc=True)
    assert np.array_equal(rt.gemm_int8(aq, bq, sa, sb, bias, 4, 0.5, 1.5), want)
    # the general form of the epilogue: accumulators too, the output transposed
    got, acc = rt.gemm_int8(aq, bq, sa, sb, bias, 4, 0.5, 1.5, output_transpose=True, want_acc=True)
    assert np.array_equal(acc, wacc) and np.array_equal(got.T, want)


@pytest.mark.parametrize("m,n,k", [(1793, 1794, 512), (1920, 1802, 576), (1799, 1792, 640), (2050, 2178, 64), (2048, 2178, 192), (2050, 2176, 256), (2050, 1986, 192), (2050, 1922, 192)])
@pytest.mark.parametrize("per_col", [True, False])
def test_128x128_tiles_cut_at_the_end(rt, m, n, k, per_col):
    """200 tiles of 128 x 128 and more with a cut last row or column of tiles, in both forms of the K step: rows past the end repeat the
    last one, and nothing is written outside the output (an odd number of columns in rows of an even stride).  (The last shape, 272 tiles but
    no more than 1024 of 64 x 64, takes those.)"""
    print("[case]", m, n, k, per_col, flush=True)
    a, bq, sb, bias = cases.gemm_case(m + n + k, m, n, k, per_col=per_col)
    aq, sa = rt.gemm_quantize_rows(a)
    want, _ = npref.gemm_int8(aq, bq, sa, sb, bias, 4, acc=npref.gemm_acc_exact(aq, bq))
    assert np.array_equal(rt.gemm_int8(aq, bq, sa, sb, bias, 4), want)
    cols = n - 1
    da, db, dsa, dsb, dc = rt.up(aq), rt.up(bq), rt.up(sa), rt.up(sb[:cols] if per_col else sb), rt.up(bias.reshape(-1)[:cols])
    out = rt.up(np.full((m + 1, n + 2), 7.0, np.float32))
    check(lib().ncnnhip_gemm_int8(da.ptr, k, db.ptr, k, m, cols, k, dsa.ptr, dsb.ptr, cols if per_col else 1, dc.ptr, 4, 1.0, 1.0, 0, out.ptr, n + 2, None, rt.stream))
    got = out.to_numpy(rt.stream)
    assert np.array_equal(got[:m, :cols], want[:, :cols]) and np.all(got[:m, cols:] == 7.0) and np.all(got[m] == 7.0)


@pytest.mark.parametrize("m,n,k", [(2945, 2900, 64), (2820, 3076, 128), (2817, 2824, 192), (3072, 2820, 256), (2821, 3072, 320), (2944, 2944, 1024), (4100, 6148, 64)])
@pytest.mark.parametrize("per_col", [True, False])
def test_256x256_tiles_cut_at_the_end(rt, m, n, k, per_col):
    """More than 512 tiles of 128 x 128 in one round of 256 x 256, and a second round that is well filled, K of one step to more than the ring holds: rows past the end
    repeat the last one, and nothing is written outside the output.  Columns that are no whole fours, and output rows off 16 bytes, take other kernels and give the same."""
    print("[case]", m, n, k, per_col, flush=True)
    a, bq, sb, bias = cases.gemm_case(m + n + k, m, n, k, per_col=per_col)
    aq, sa = rt.gemm_quantize_rows(a)
    want, _ = npref.gemm_int8(aq, bq, sa, sb, bias, 4, acc=npref.gemm_acc_exact(aq, bq))
    assert np.array_equal(rt.gemm_int8(aq, bq, sa, sb, bias, 4), want)
    da, db, dsa, dsb, dc = rt.up(aq), rt.up(bq), rt.up(sa), rt.up(sb), rt.up(bias.reshape(-1))
    for cols, stride in ((n - 4, n + 4), (n - 5, n), (n, n + 2)):
        out = rt.up(np.full((m + 1, stride), 7.0, np.float32))
        check(lib().ncnnhip_gemm_int8(da.ptr, k, db.ptr, k, m, cols, k, dsa.ptr, dsb.ptr, cols if per_col else 1, dc.ptr, 4, 1.0, 1.0, 0, out.ptr, stride, None, rt.stream))
        got = out.to_numpy(rt.stream)
        assert np.array_equal(got[:m, :cols], want[:, :cols]) and np.all(got[:m, cols:] == 7.0) and np.all(got[m] == 7.0)


@pytest.mark.parametrize("a_stride,o_stride", [(64, (1 << 20) + 4), ((1 << 24) + 16, 32768)])
@pytest.mark.parametrize("per_col", [True, False])
def test_256x256_tiles_of_rows_far_apart(rt, a_stride, o_stride, per_col):
    """128 whole tiles of one K step whose output rows are more than 2^20 floats apart, or whose 256 rows of A take more than 4 GiB: offsets inside a tile
    beyond 32 bits.  Nothing is written between the rows."""
    print("[case]", a_stride, o_stride, per_col, flush=True)
    m, n, k = 256, 32768, 64
    a, bq, sb, bias = cases.gemm_case(a_stride % 1000, m, n, k, per_col=per_col)
    aq, sa = rt.gemm_quantize_rows(a)
    want, _ = npref.gemm_int8(aq, bq, sa, sb, bias, 4, acc=npref.gemm_acc_exact(aq, bq))
    da, db, dsa, dsb, dc = DeviceBuffer((m - 1) * a_stride + k), rt.up(bq), rt.up(sa), rt.up(sb), rt.up(bias.reshape(-1))
    for i in range(m):
        check(lib().ncnnhip_memcpy_h2d(C.c_void_p(da.ptr.value + i * a_stride), aq[i].ctypes.data_as(C.c_void_p), k, rt.stream))
    check(lib().ncnnhip_stream_synchronize(rt.stream))
    out = rt.up(np.full((m, o_stride), 7.0, np.float32))
    check(lib().ncnnhip_gemm_int8(da.ptr, a_stride, db.ptr, k, m, n, k, dsa.ptr, dsb.ptr, n if per_col else 1, dc.ptr, 4, 1.0, 1.0, 0, out.ptr, o_stride, None, rt.stream))
    got = out.to_numpy(rt.stream)
    assert np.array_equal(got[:, :n], want) and np.all(got[:, n:] == 7.0)


@pytest.mark.parametrize("m,n,k,pad", [(1601, 1537, 1003, 0), (1850, 1800, 1004, 0), (1793, 1805, 1024, 1), (2305, 2241, 1002, 2)])
def test_128x128_tiles_of_rows_off_16_bytes(rt, m, n, k, pad):
    """Rows that begin at any byte, or at any fourth, in the sizes that take 128 x 128 tiles for it: cut tiles, K that ends inside a step."""
    print("[case]", m, n, k, pad, flush=True)
    a, bq, sb, bias = cases.gemm_case(m + n + k, m, n, k, per_col=True)
    aq, sa = rt.gemm_quantize_rows(a)
    want, _ = npref.gemm_int8(aq, bq, sa, sb, bias, 4, acc=npref.gemm_acc_exact(aq, bq))
    wide = np.full((m, k + pad), 99, np.int8)
    wide[:, :k] = aq
    da, db, dsa, dsb, dc = rt.up(wide), rt.up(bq), rt.up(sa), rt.up(sb), rt.up(bias.reshape(-1))
    out = rt.up(np.full((m + 1, n + 1), 7.0, np.float32))
    check(lib().ncnnhip_gemm_int8(da.ptr, k + pad, db.ptr, k, m, n, k, dsa.ptr, dsb.ptr, n, dc.ptr, 4, 1.0, 1.0, 0, out.ptr, n + 1, None, rt.stream))
    got = out.to_numpy(rt.stream)
    assert np.array_equal(got[:m, :n], want) and np.all(got[:m, n] == 7.0) and np.all(got[m] == 7.0)
