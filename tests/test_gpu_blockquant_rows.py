"""Block-quantised Gemm on many activation rows: groups of 16 rows, tiles of 16 weight rows and the K steps of 64 at
their edges, every packed layout, alone and with several matrices in one call: against the oracle and a float64 value."""
import ctypes as C

import numpy as np
import pytest

from ncnn_amd import synth
from ncnn_amd.hip import DeviceBuffer, check, lib
from oracle import oracle
from tests import npref

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module")
def rt():
    import ncnn_amd
    return ncnn_amd.Runtime(0)


def _check(got, a, packed, scales, bits, block, c=None, bt=-1, alpha=1.0, beta=1.0):
    # every product q * a is exact; what differs from the references is the order of the fp32 additions (see the random walk)
    val, floor = npref.blockquant_gemm_f64(a, packed, scales, bits, block, None, c, bt, alpha, beta)
    ref = oracle.gemm_blockquant(a, packed, scales, bits, block, None, c, bt, alpha, beta)
    tol = 1e-5 * floor + 1e-30
    assert np.all(np.abs(got - ref) <= tol) and np.all(np.abs(got - val) <= tol)


@pytest.mark.parametrize("m,n,k", [(17, 15, 16), (32, 16, 64), (33, 17, 80), (48, 200, 512), (49, 65, 576), (64, 130, 1040), (65, 33, 192), (130, 96, 128), (18, 4200, 256)])
@pytest.mark.parametrize("bits,block", [(8, 64), (8, 32), (6, 128), (6, 32), (4, 64), (4, 32)])
def test_many_fp16_rows(rt, m, n, k, bits, block):
    print("[case]", m, n, k, bits, block, flush=True)
    a, packed, scales = synth.blockquant_operands(m + n + k, m, n, k, bits, block)
    c = np.random.default_rng(n).normal(size=(1, n)).astype(F)
    pw, pd = rt.blockquant_pack(packed, scales, block, bits=bits, k=k)
    got = rt.gemm_blockquant_packed(a.astype(np.float16), pw, pd, n, c, 4, 0.75, 1.5, bits=bits, block=block)
    _check(got, a, packed, scales, bits, block, c, 4, 0.75, 1.5)


@pytest.mark.parametrize("m,n,k", [(64, 17610, 144), (50, 16800, 336)])
@pytest.mark.parametrize("bits,block", [(8, 64), (8, 32), (6, 128), (6, 32), (4, 64), (4, 32)])
def test_four_groups_of_rows_and_six_tiles(rt, m, n, k, bits, block):
    """The largest form, which has the fewest registers to spare: blocks of 32 read a tile's descales while the one before is multiplied."""
    test_many_fp16_rows(rt, m, n, k, bits, block)


@pytest.mark.parametrize("m,n,k,bits,block", [(5, 40, 8208, 4, 64), (13, 33, 9216, 6, 32), (16, 20, 8704, 8, 32), (5, 19600, 1024, 4, 128), (7, 7000, 9200, 8, 64)])
def test_few_fp16_rows_of_large_weights(rt, m, n, k, bits, block):
    test_many_fp16_rows(rt, m, n, k, bits, block)


@pytest.mark.parametrize("m,n,k", [(20, 33, 80), (40, 16, 528), (66, 200, 1072), (17, 20, 48), (9, 20, 9168), (16, 400, 9200),
                                   (3, 20, 80), (5, 16, 192), (9, 40, 1072), (9, 4100, 1072), (16, 20, 4112), (5, 20, 8208), (9, 520, 8208), (3, 40, 9200)])
@pytest.mark.parametrize("bits,block", [(8, 64), (8, 32), (6, 64), (4, 32), (4, 128)])
def test_an_infinity_stays_an_infinity(rt, m, n, k, bits, block):
    """K ends inside a step of 64, or a wavefront has fewer steps than its neighbours: what is read in place of the values beyond
    its share is the start of the row or of the share, and must not count.
    With no other special value and no zero weight in its column, an infinite activation gives infinities and no NaN."""
    print("[case]", m, n, k, bits, block, flush=True)
    a, packed, scales = synth.blockquant_operands(m + n + k, m, n, k, bits, block)
    a = a.astype(np.float16)
    a[0, 0], a[1, 7], a[2, k - 1] = np.inf, -np.inf, np.inf
    with np.errstate(invalid="ignore"):
        want = oracle.gemm_blockquant(a.astype(F), packed, scales, bits, block)
    pw, pd = rt.blockquant_pack(packed, scales, block, bits=bits, k=k)
    got = rt.gemm_blockquant_packed(a, pw, pd, n, bits=bits, block=block)
    assert np.array_equal(np.isnan(got[:3]), np.isnan(want[:3])) and np.isinf(want[:3]).any()
    inf = np.isinf(want[:3])
    assert np.array_equal(got[:3][inf], want[:3][inf])
    _check(got[3:], a[3:].astype(F), packed, scales, bits, block)


@pytest.mark.parametrize("m", [17, 40, 100])
def test_several_matrices_in_one_call(rt, m):
    k, ns = 192, (50, 16, 700)
    ops = [synth.blockquant_operands(10 + i, m, n, k, 4, 64) for i, n in enumerate(ns)]
    a = ops[0][0]
    mats = [rt.blockquant_pack(p, s, 64, bits=4, k=k) + (n, None, -1, 1.0, 1.0) for (_, p, s), n in zip(ops, ns)]
    outs = rt.gemm_blockquant_packed_multi(a.astype(np.float16), mats, bits=4, block=64)
    for (_, p, s), got in zip(ops, outs):
        _check(got, a, p, s, 4, 64)


@pytest.mark.parametrize("m,n,k", [(129, 16, 16), (130, 72, 144), (191, 33, 64), (200, 1000, 1040), (1025, 1000, 320), (1025, 1000, 1552), (1024, 2048, 96), (1030, 2050, 128)])
@pytest.mark.parametrize("bits,block", [(8, 64), (8, 32), (6, 128), (6, 32), (4, 64), (4, 32)])
def test_many_fp32_rows(rt, m, n, k, bits, block):
    """Both tile widths of the kernel that splits K inside a workgroup and the kernel beyond it: one K step (the second
    half has none), odd and even numbers of steps, tiles beyond the last row and weight row."""
    print("[case]", m, n, k, bits, block, flush=True)
    a, packed, scales = synth.blockquant_operands(m + n + k, m, n, k, bits, block)
    c = np.random.default_rng(n).normal(size=(m, n)).astype(F)
    pw, pd = rt.blockquant_pack(packed, scales, block, bits=bits, k=k)
    got = rt.gemm_blockquant_packed(a, pw, pd, n, c, 3, 0.75, 1.5, bits=bits, block=block, rows_kernel=True)
    _check(got, a, packed, scales, bits, block, c, 3, 0.75, 1.5)


@pytest.mark.parametrize("m,n,k,rows", [(1, 33, 80, False), (4, 20, 528, False), (9, 16, 1072, False), (5, 20, 80, True), (20, 33, 1072, True), (40, 16, 8208, True),
                                        (70, 200, 528, True), (200, 1000, 1040, True)])
@pytest.mark.parametrize("bits,block", [(8, 64), (8, 32), (6, 64), (4, 32)])
def test_an_infinity_stays_an_infinity_fp32(rt, m, n, k, rows, bits, block):
    """The same for fp32 rows: the one-pass form, the 16-row passes and the tiles of 64 rows."""
    print("[case]", m, n, k, rows, bits, block, flush=True)
    a, packed, scales = synth.blockquant_operands(m + n + k, m, n, k, bits, block, half_exact=False)
    a[0, 0], a[m // 2, k - 1] = np.inf, -np.inf
    with np.errstate(invalid="ignore"):
        want = oracle.gemm_blockquant(a, packed, scales, bits, block)
    pw, pd = rt.blockquant_pack(packed, scales, block, bits=bits, k=k)
    got = rt.gemm_blockquant_packed(a, pw, pd, n, bits=bits, block=block, **({"rows_kernel": True} if rows else {}))
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.isinf(want).any()
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf])


# (m, n): every pair of 1 or 2 groups of rows and 1 to 4 tiles a workgroup, with rows and weight rows that fill neither
@pytest.mark.parametrize("m,n,k", [(5, 33, 80), (16, 16, 64), (5, 4100, 80), (9, 8200, 144), (5, 13000, 80), (17, 8200, 80), (20, 12410, 64), (130, 50, 1040), (547, 137, 64), (40, 300, 592)])
@pytest.mark.parametrize("bits,block", [(8, 64), (8, 32), (6, 128), (6, 32), (4, 64), (4, 32)])
@pytest.mark.parametrize("rows", [False, True])
def test_fp32_rows_split_as_they_are_multiplied(rt, m, n, k, bits, block, rows):
    print("[case]", m, n, k, bits, block, rows, flush=True)
    a, packed, scales = synth.blockquant_operands(m + n + k, m, n, k, bits, block, half_exact=False)
    rng = np.random.default_rng(n)
    c, ins = rng.normal(size=(m, n)).astype(F), rng.uniform(0.5, 1.5, k).astype(F)
    pw, pd = rt.blockquant_pack(packed, scales, block, bits=bits, k=k)
    got = rt.gemm_blockquant_packed(a, pw, pd, n, c, 3, 0.75, 1.5, bits=bits, block=block, in_scales=ins, rows_kernel=rows)
    val, floor = npref.blockquant_gemm_f64(a, packed, scales, bits, block, ins, c, 3, 0.75, 1.5)
    assert np.all(np.abs(got - val) <= 1e-5 * floor + 1e-30)
    got = rt.gemm_blockquant_packed(a, pw, pd, n, bits=bits, block=block, rows_kernel=rows)
    val, floor = npref.blockquant_gemm_f64(a, packed, scales, bits, block)
    assert np.all(np.abs(got - val) <= 1e-5 * floor + 1e-30)


@pytest.mark.parametrize("m,n,k", [(32, 14330, 144), (25, 11000, 208), (32, 16100, 592)])
@pytest.mark.parametrize("bits,block", [(8, 64), (8, 32), (6, 128), (6, 32), (4, 64), (4, 32)])
def test_two_groups_of_fp32_rows_and_three_or_four_tiles(rt, m, n, k, bits, block):
    """The largest forms for fp32 rows, which go tile by tile; blocks of 32 read a tile's descales while the one before is multiplied."""
    test_fp32_rows_split_as_they_are_multiplied(rt, m, n, k, bits, block, True)


@pytest.mark.parametrize("m,n,k", [(7, 40, 144), (17, 8200, 80)])
def test_special_values_in_fp32_rows(rt, m, n, k):
    """The sums are made without a look at the values and repeated with one where they turn out not to be numbers: infinities, the largest
    finite value and a NaN must give what the careful split gives, also beside an input scale, also in the padding of a ragged K."""
    a, packed, scales = synth.blockquant_operands(m + n, m, n, k, 8, 64, half_exact=False)
    a[0, 0], a[2, k - 1], a[3, 1], a[4, 2] = np.inf, -np.inf, np.finfo(F).max * F(1e-3), np.nan
    ins = np.ones(k, F)
    ins[0] = 2.0
    pw, pd = rt.blockquant_pack(packed, scales, 64, k=k)
    with np.errstate(invalid="ignore", over="ignore"):
        want = oracle.gemm_blockquant(a, packed, scales, 8, 64, ins)
    got = rt.gemm_blockquant_packed(a, pw, pd, n, in_scales=ins)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.isinf(want[0]).any() and np.isnan(want[4]).all()
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf])
    fine = np.isfinite(want)
    val, floor = npref.blockquant_gemm_f64(np.where(np.isfinite(a), a, 0), packed, scales, 8, 64, ins)
    rows = [i for i in range(m) if i not in (0, 2, 4)]
    assert np.all(np.abs(got[rows] - val[rows])[fine[rows]] <= 1e-5 * floor[rows][fine[rows]])


def test_fp32_rows_off_16_bytes_take_the_general_forms(rt):
    """packed_rows takes activations and outputs of any 4-byte alignment: what the aligned call gives, to the order of the sums."""
    m, n, k = 24, 100, 208
    a, packed, scales = synth.blockquant_operands(5, m, n, k, 4, 64, half_exact=False)
    pw, pd = rt.blockquant_pack(packed, scales, 64, bits=4, k=k)
    w, d = rt.up(pw), rt.up(pd)
    size = C.c_size_t()
    check(lib().ncnnhip_gemm_blockquant_packed_rows_workspace_bytes(m, k, C.byref(size)))
    ws = DeviceBuffer.empty((size.value,), np.uint8)
    val, floor = npref.blockquant_gemm_f64(a, packed, scales, 4, 64)
    for a_stride, a_off, o_stride, o_off in ((k, 0, n, 0), (k + 1, 0, n + 1, 0), (k + 4, 1, n + 4, 1), (k + 4, 0, n + 4, 2), (k + 3, 3, n + 3, 3)):
        buf = np.full(m * a_stride + 8, np.nan, F)
        buf[a_off:a_off + m * a_stride].reshape(m, a_stride)[:, :k] = a
        src, dst = rt.up(buf), rt.up(np.full(m * o_stride + 8, 7.0, F))
        at = lambda t, off: C.c_void_p(t.ptr.value + 4 * off)
        check(lib().ncnnhip_gemm_blockquant_packed_rows(at(src, a_off), a_stride, m, n, k, w.ptr, d.ptr, 4, 64, None, None, -1, 1.0, 1.0, at(dst, o_off), o_stride, ws.ptr,
                                                        size.value, rt.stream))
        out = dst.to_numpy(rt.stream)
        got = out[o_off:o_off + m * o_stride].reshape(m, o_stride)
        assert np.all(np.abs(got[:, :n] - val) <= 1e-5 * floor), (a_stride, a_off)
        assert np.all(got[:, n:] == 7.0) and np.all(out[:o_off] == 7.0), (o_stride, o_off)


@pytest.mark.parametrize("m,k,ns", [(3, 144, (50, 16, 4200)), (4, 4112, (50, 16, 4200)), (9, 208, (50, 16, 4200)), (16, 1040, (50, 16, 4200)), (17, 208, (50, 16, 4200)),
                                    # groups of three tiles would be 256 only if they went across matrices: groups of four, and padding to whole eights
                                    (5, 1040, (4096,) * 3), (16, 2064, (4096, 4090, 4081)), (13, 208, (1000,) * 8)])
def test_several_matrices_of_fp32_rows_get_the_bits_of_single_calls(rt, m, k, ns):
    ops = [synth.blockquant_operands(10 + i, m, n, k, 8, 64, half_exact=False) for i, n in enumerate(ns)]
    a = ops[0][0]
    mats = [rt.blockquant_pack(p, s, 64, k=k) + (n, None, -1, 1.0, 1.0) for (_, p, s), n in zip(ops, ns)]
    for got, (pw, pd, n, *_) in zip(rt.gemm_blockquant_packed_multi(a, mats), mats):
        assert np.array_equal(got, rt.gemm_blockquant_packed(a, pw, pd, n))


@pytest.mark.parametrize("m,n,k", [(1030, 1000, 16), (1100, 1000, 64), (1030, 970, 80), (523, 1960, 144), (65, 8250, 208), (1025, 1010, 320), (260, 3300, 1040), (1090, 960, 1568),
                                   (2060, 2050, 80), (2830, 1530, 144)])
@pytest.mark.parametrize("bits,block", [(8, 64), (8, 128), (6, 64), (4, 128)])
def test_fp32_rows_in_64x128_tiles(rt, m, n, k, bits, block):
    """More than 256 tiles of 64 x 64 (in the last two shapes the plain layout takes 64 x 192 ones): row blocks and weight tiles cut off, K groups of no, one and several steps, the last of them ragged;
    with input scales and C, rows off 16 bytes, an infinity and a NaN (no special value beyond its own row)."""
    print("[case]", m, n, k, bits, block, flush=True)
    a, packed, scales = synth.blockquant_operands(m + n + k, m, n, k, bits, block, half_exact=False)
    rng = np.random.default_rng(n)
    c, ins = rng.normal(size=(m, n)).astype(F), rng.uniform(0.5, 2.0, k).astype(F)
    pw, pd = rt.blockquant_pack(packed, scales, block, bits=bits, k=k)
    got = rt.gemm_blockquant_packed(a, pw, pd, n, c, 3, 0.75, 1.5, bits=bits, block=block, in_scales=ins, rows_kernel=True)
    val, floor = npref.blockquant_gemm_f64(a, packed, scales, bits, block, ins, c, 3, 0.75, 1.5)
    assert np.all(np.abs(got - val) <= 1e-5 * floor + 1e-30)

    w, d = rt.up(pw), rt.up(pd)
    size = C.c_size_t()
    check(lib().ncnnhip_gemm_blockquant_packed_rows_workspace_bytes(m, k, C.byref(size)))
    ws = DeviceBuffer.empty((size.value,), np.uint8)
    a[1, k - 1], a[m - 1, 0] = np.inf, np.nan
    buf = np.full(m * (k + 3) + 8, np.nan, F)
    buf[1:1 + m * (k + 3)].reshape(m, k + 3)[:, :k] = a
    src, dst = rt.up(buf), rt.up(np.full(m * (n + 1) + 8, 7.0, F))
    check(lib().ncnnhip_gemm_blockquant_packed_rows(C.c_void_p(src.ptr.value + 4), k + 3, m, n, k, w.ptr, d.ptr, bits, block, None, None, -1, 1.0, 1.0,
                                                    C.c_void_p(dst.ptr.value + 4), n + 1, ws.ptr, size.value, rt.stream))
    out = dst.to_numpy(rt.stream)
    got = out[1:1 + m * (n + 1)].reshape(m, n + 1)
    assert np.all(got[:, n] == 7.0) and out[0] == 7.0 and np.all(out[1 + m * (n + 1):] == 7.0)
    rows = [i for i in range(m) if i not in (1, m - 1)]
    val, floor = npref.blockquant_gemm_f64(a[rows], packed, scales, bits, block)
    assert np.all(np.abs(got[rows, :n] - val) <= 1e-5 * floor + 1e-30)
    q = npref.blockquant_gemm_f64(np.eye(k, dtype=F)[k - 1:], packed, scales, bits, block)[0][0]  # the weights that meet the infinity
    assert np.array_equal(got[1, :n][q != 0], np.where(q > 0, np.inf, -np.inf)[q != 0].astype(F)) and np.all(np.isnan(got[1, :n][q == 0])) and np.all(np.isnan(got[m - 1, :n]))


@pytest.mark.parametrize("m,n,k,bits", [(130, 40, 4112, 8), (133, 130, 12304, 4), (129, 16, 12816, 8), (140, 24, 144, 6),  # few tiles: K over two groups of wavefronts
                                        (1030, 1010, 400, 8), (1090, 960, 144, 4), (1030, 1000, 208, 6),                         # 64 x 128 tiles
                                        (2060, 2050, 144, 8)])                                                                  # 64 x 192
def test_fp32_rows_of_any_magnitude(rt, m, n, k, bits):
    """Rows of zeros, of subnormals, as large as a K step holds, with few values of any weight, and rows whose largest values meet weights of zero: an activation keeps its 24 bits
    whatever stands beside it (of the least of its three bf16 numbers, what lies above 2^-134), so that the sums' roundings are the only error.  A step adds up to 64 products
    with fields of up to 127 before their scale: less than 2^13 times the largest activation, so that magnitudes up to 2^114 stay below 2^127 (every form has this limit)."""
    a, packed, scales = synth.blockquant_operands(m + n, m, n, k, bits, 64, half_exact=False)
    rng = np.random.default_rng(k)
    scales *= 64  # outputs of the largest row stay finite
    a[0] = 0
    a[1], a[2], a[3] = a[1] * F(2.0 ** -130), a[2] * F(2.0 ** -112), a[3] * F(2.0 ** 114) / max(1, np.abs(a[3]).max())
    a[4] *= np.exp2(rng.integers(-60, 60, k)).astype(F)
    a[5, 1:] *= F(2.0 ** -35)
    a[m - 1, : k - 1] = 0
    a[6, 64:80] *= F(2.0 ** 50)  # a field of zero whatever its block's scale: these columns weigh nothing
    a[7, 64:80] = F(2.0 ** 100)
    packed[:, 64 * bits // 8:80 * bits // 8] = 0
    pw, pd = rt.blockquant_pack(packed, scales, 64, bits=bits, k=k)
    w, d = rt.up(pw), rt.up(pd)
    size = C.c_size_t()
    check(lib().ncnnhip_gemm_blockquant_packed_rows_workspace_bytes(m, k, C.byref(size)))
    ws = DeviceBuffer.empty((size.value,), np.uint8)
    src, dst = rt.up(np.concatenate([[F(0)], a.ravel()]).astype(F)), rt.up(np.full((m, n), 7.0, F))
    check(lib().ncnnhip_gemm_blockquant_packed_rows(C.c_void_p(src.ptr.value + 4), k, m, n, k, w.ptr, d.ptr, bits, 64, None, None, -1, 1.0, 1.0, dst.ptr, n,
                                                    ws.ptr, size.value, rt.stream))  # (off 16 bytes: not the one-launch form)
    got = dst.to_numpy(rt.stream)
    val, floor = npref.blockquant_gemm_f64(a, packed, scales, bits, 64)
    assert np.all(np.isfinite(got)) and np.all(got[0] == 0)
    ones = npref.blockquant_gemm_f64(np.ones((1, k), F), packed, scales, bits, 64)[1]
    assert np.all(np.abs(got - val) <= 1e-6 * floor + 2.0 ** -133 * ones)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m,k", [(129, 64), (191, 272), (131, 4096), (131, 4112), (193, 8192), (131, 8208), (131, 12288), (193, 12304)])
def test_split_pass_of_rows_of_their_own_size(rt, m, k, bits):
    """Every row has its own size, so that a row or a piece of one out of place shows, on K of one step to many and a part of one.  The bound is that of
    test_fp32_rows_of_any_magnitude: the sums' roundings, relative to the sum of magnitudes."""
    a, packed, scales = synth.blockquant_operands(m + k, m, 48, k, bits, 64, half_exact=False)
    a *= np.exp2(np.arange(m) % 41 - 20).astype(F)[:, None]
    pw, pd = rt.blockquant_pack(packed, scales, 64, bits=bits, k=k)
    w, d = rt.up(pw), rt.up(pd)
    size = C.c_size_t()
    check(lib().ncnnhip_gemm_blockquant_packed_rows_workspace_bytes(m, k, C.byref(size)))
    ws = DeviceBuffer.empty((size.value,), np.uint8)
    src, dst = rt.up(np.concatenate([[F(0)], a.ravel()]).astype(F)), rt.up(np.full((m, 48), 7.0, F))
    check(lib().ncnnhip_gemm_blockquant_packed_rows(C.c_void_p(src.ptr.value + 4), k, m, 48, k, w.ptr, d.ptr, bits, 64, None, None, -1, 1.0, 1.0, dst.ptr, 48,
                                                    ws.ptr, size.value, rt.stream))  # (off 16 bytes: not the one-launch form)
    val, floor = npref.blockquant_gemm_f64(a, packed, scales, bits, 64)
    assert np.all(np.abs(dst.to_numpy(rt.stream) - val) <= 1e-6 * floor)


def test_several_matrices_whose_groups_would_fill_the_units_only_together(rt):
    """3 x 256 tiles: in groups of three 258, in groups of four 192, which is what several matrices get; one matrix of all of them is 256 groups of three."""
    m, k, n = 48, 64, 4096
    ops = [synth.blockquant_operands(30 + i, m, n, k, 4, 64) for i in range(3)]
    a = ops[0][0].astype(np.float16)
    mats = [rt.blockquant_pack(p, s, 64, bits=4, k=k) + (n, None, -1, 1.0, 1.0) for _, p, s in ops]
    for got, (_, packed, scales) in zip(rt.gemm_blockquant_packed_multi(a, mats, bits=4, block=64), ops):
        _check(got, a.astype(F), packed, scales, 4, 64)


@pytest.mark.parametrize("m,k,ns,bits,block", [
    # the form of all matrices shares K out over fewer wavefronts than the one each matrix gets alone: 8 bits 8 and 7, 4 bits 8 and 7, 8 and 6
    (48, 528, (4096,) * 3, 8, 64), (64, 512, (4096,) * 3, 4, 64), (64, 592, (11008,) * 2, 4, 32), (48, 512, (11008,) * 2, 8, 64),
    # matrices that alone get different numbers of wavefronts
    (64, 512, (4096, 11008), 8, 64), (57, 512, (16, 4096, 17600), 4, 64),
    # 5 to 16 rows: small weights alone go to another kernel than all of them
    (16, 4096, (4096,) * 2, 4, 64), (7, 4096, (4096,) * 2, 6, 32), (5, 4096, (4096, 8192), 4, 64), (16, 8208, (2000, 6000), 8, 64), (16, 4096, (4096, 7200), 8, 32), (9, 1040, (16400, 64), 8, 64),
    # up to 4 rows the same bits whatever the sizes
    (4, 4096, (4096,) * 3, 4, 64), (3, 8208, (2000, 18000), 8, 64), (1, 1040, (16400, 64), 6, 32), (2, 4112, (40, 11008), 8, 128)])
def test_several_matrices_of_fp16_rows_beside_single_calls(rt, m, k, ns, bits, block):
    """Where the size of the whole launch asks for another kernel, or another split of K, than that of one matrix: the results differ by
    the order of the additions only, and not at all up to four rows."""
    print("[case]", m, k, ns, bits, block, flush=True)
    ops = [synth.blockquant_operands(40 + i, m, n, k, bits, block) for i, n in enumerate(ns)]
    a = ops[0][0].astype(np.float16)
    mats = [rt.blockquant_pack(p, s, block, bits=bits, k=k) + (n, None, -1, 1.0, 1.0) for (_, p, s), n in zip(ops, ns)]
    for got, (pw, pd, n, *_), (_, packed, scales) in zip(rt.gemm_blockquant_packed_multi(a, mats, bits=bits, block=block), mats, ops):
        single = rt.gemm_blockquant_packed(a, pw, pd, n, bits=bits, block=block)
        val, floor = npref.blockquant_gemm_f64(a.astype(F), packed, scales, bits, block)
        tol = 1e-5 * floor + 1e-30  # as _check
        assert np.all(np.abs(got - val) <= tol) and np.all(np.abs(single - val) <= tol), n
        assert m > 4 or np.array_equal(got, single), n
