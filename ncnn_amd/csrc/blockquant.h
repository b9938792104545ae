// Block-quantised weights: how packed fields become matrix-core operands, and the description of several matrices that share
// their activation rows.  Used by the kernels of blockquant.hip and blockquant_rows.hip.
#ifndef NCNNHIP_BLOCKQUANT_H
#define NCNNHIP_BLOCKQUANT_H

#include <hip/hip_fp16.h>

#include "common.h"

namespace ncnnhip {

typedef int v4i_bq __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float load_c(const float* c, int bt, int i, int j, int N)
{
    if (bt == 0) return c[0];
    if (bt == 1 || bt == 2) return c[i];
    if (bt == 3) return c[(size_t)i * N + j];
    return c[j];
}

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));

__device__ __forceinline__ v8h bytes_to_halves(int lo, int hi)
{
    // lo, hi: 8 bytes u0..u7 (u = q + 128).  Build halves 0x6400|u = 1024+u, then subtract 1152.
    union
    {
        int i[4];
        v2h h2[4];
        v8h h8;
    } t;
    t.i[0] = __builtin_amdgcn_perm(0x64646464, lo, 0x04010400);
    t.i[1] = __builtin_amdgcn_perm(0x64646464, lo, 0x04030402);
    t.i[2] = __builtin_amdgcn_perm(0x64646464, hi, 0x04010400);
    t.i[3] = __builtin_amdgcn_perm(0x64646464, hi, 0x04030402);
    const v2h off = {(_Float16)1152.f, (_Float16)1152.f};
#pragma unroll
    for (int e = 0; e < 4; e++) t.h2[e] = t.h2[e] - off;
    return t.h8;
}

// (x & mask) | bits in one instruction, which takes one of its constants from a scalar register (the compiler makes two instructions with
// literals of it)
__device__ __forceinline__ unsigned and_or(unsigned x, unsigned mask, unsigned bits)
{
    unsigned r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(mask), "v"(bits));
    return r;
}

// 8 nibbles u = q + 8; nibbles p and p + 4 of the dword are the two halves of pair p, so one mask serves both.  A nibble at bit 0 of
// a half makes 1024 + u with the exponent of 1024 above it, one at bit 4 makes 64 + u with that of 64: one shift for the dword,
// nine instructions where shifting and masking every pair took fifteen (us before and after: 48 rows of 4096 x 11008 17.7 15.9,
// 96 of 11008 x 4096 20.8 18.7, 16 of 22016 x 4096 14.4 13.0, one of 4096 x 11008 7.9 7.4).
__device__ __forceinline__ v8h nibbles_to_halves(unsigned w)
{
    union
    {
        unsigned i[4];
        v2h h2[4];
        v8h h8;
    } t;
    const unsigned v = w >> 8;
    t.i[0] = and_or(w, 0x000F000Fu, 0x64006400u);
    t.i[1] = and_or(w, 0x00F000F0u, 0x54005400u);
    t.i[2] = and_or(v, 0x000F000Fu, 0x64006400u);
    t.i[3] = and_or(v, 0x00F000F0u, 0x54005400u);
    const v2h off0 = {(_Float16)1032.f, (_Float16)1032.f}, off4 = {(_Float16)72.f, (_Float16)72.f};
#pragma unroll
    for (int e = 0; e < 4; e++) t.h2[e] = t.h2[e] - (e & 1 ? off4 : off0);
    return t.h8;
}

// 16 six-bit fields u = q + 32 in three dwords.  A dword carries two whole pairs (the low-half field at bit 0 or 6,
// the high-half field 16 bits above) and, in bits 12-15 / 28-31, a third of a pair: pairs 6 and 7 have their low four
// bits in dword 0 / dword 1 and their high two bits side by side in dword 2.
__device__ __forceinline__ void sixbit_to_halves(unsigned d0, unsigned d1, unsigned d2, v8h& wa, v8h& wb)
{
    union
    {
        unsigned i[4];
        v2h h2[4];
        v8h h8;
    } a, b;
    const unsigned magic = 0x64006400u;
    a.i[0] = and_or(d0, 0x003F003Fu, magic);
    a.i[1] = and_or(d0 >> 6, 0x003F003Fu, magic);
    a.i[2] = and_or(d1, 0x003F003Fu, magic);
    a.i[3] = and_or(d1 >> 6, 0x003F003Fu, magic);
    b.i[0] = and_or(d2, 0x003F003Fu, magic);
    b.i[1] = and_or(d2 >> 6, 0x003F003Fu, magic);
    b.i[2] = and_or(d0 >> 12, 0x000F000Fu, and_or(d2 >> 8, 0x00300030u, magic));
    b.i[3] = and_or(d1 >> 12, 0x000F000Fu, and_or(d2 >> 10, 0x00300030u, magic));
    const v2h off = {(_Float16)1056.f, (_Float16)1056.f};
#pragma unroll
    for (int e = 0; e < 4; e++)
    {
        a.h2[e] = a.h2[e] - off;
        b.h2[e] = b.h2[e] - off;
    }
    wa = a.h8;
    wb = b.h8;
}

typedef int v2i_bq __attribute__((ext_vector_type(2)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

__device__ __forceinline__ void split_bf16x3(float v, unsigned& hi, unsigned& mid, unsigned& lo) // each in the upper half of its dword
{
    const unsigned b = __float_as_uint(v);
    hi = b & 0xFFFF0000u;
    const bool finite = (b & 0x7F800000u) != 0x7F800000u; // infinities and NaNs travel in hi alone
    const float r1 = finite ? v - __uint_as_float(hi) : 0.f;
    mid = __float_as_uint(r1) & 0xFFFF0000u;
    const float r2 = r1 - __uint_as_float(mid);
    lo = __float_as_uint(r2) & 0xFFFF0000u; // at most 8 significant bits are left
}

__device__ __forceinline__ unsigned bf16_pair(float even, float odd) // both exactly representable: truncation loses nothing
{
    return __builtin_amdgcn_perm(__float_as_uint(odd), __float_as_uint(even), 0x07060302u);
}

// the 8 fields that bytes_to_halves / nibbles_to_halves / sixbit_to_halves turn into halves, as bf16
__device__ __forceinline__ v8bf bytes_to_bf16(unsigned lo, unsigned hi)
{
    union
    {
        unsigned i[4];
        v8bf h;
    } t;
    const unsigned slo = lo ^ 0x80808080u, shi = hi ^ 0x80808080u; // q + 128 -> q as a signed byte
#pragma unroll
    for (int p = 0; p < 2; p++)
    {
        t.i[p] = bf16_pair((float)(signed char)(slo >> (16 * p)), (float)(signed char)(slo >> (16 * p + 8)));
        t.i[2 + p] = bf16_pair((float)(signed char)(shi >> (16 * p)), (float)(signed char)(shi >> (16 * p + 8)));
    }
    return t.h;
}
__device__ __forceinline__ v8bf nibbles_to_bf16(unsigned w)
{
    union
    {
        unsigned i[4];
        v8bf h;
    } t;
    const unsigned x = w ^ 0x88888888u; // q + 8 -> q as a two's complement nibble: one signed bit-field extract each
#pragma unroll
    for (int p = 0; p < 4; p++) t.i[p] = bf16_pair((float)((int)(x << (28 - 4 * p)) >> 28), (float)((int)(x << (12 - 4 * p)) >> 28));
    return t.h;
}
__device__ __forceinline__ void sixbit_to_bf16(unsigned d0, unsigned d1, unsigned d2, v8bf& wa, v8bf& wb)
{
    union
    {
        unsigned i[4];
        v8bf h;
    } a, b;
    // q + 32 -> q in two's complement: flip bit 5 of every field (for pairs 6 and 7 that bit sits in dword 2's top nibbles)
    const unsigned d[3] = {d0 ^ 0x08200820u, d1 ^ 0x08200820u, d2 ^ 0xA820A820u};
#pragma unroll
    for (int P = 0; P < 8; P++)
    {
        float f[2];
#pragma unroll
        for (int h = 0; h < 2; h++)
        {
            int q;
            if (P < 6)
                q = (int)(d[P >> 1] << (26 - 6 * (P & 1) - 16 * h)) >> 26; // a signed bit-field extract
            else
            {
                const unsigned u = ((d[P - 6] >> (12 + 16 * h)) & 15u) | (((d[2] >> (12 + 2 * (P - 6) + 16 * h)) & 3u) << 4);
                q = (int)(u << 26) >> 26;
            }
            f[h] = (float)q;
        }
        (P < 4 ? a.i[P & 3] : b.i[P & 3]) = bf16_pair(f[0], f[1]);
    }
    wa = a.h;
    wb = b.h;
}

// Several weight matrices that share the activation rows, K and the field format in ONE launch (the gate and up projections of a
// decoder layer, q / k / v of an attention layer): the tiles of matrix i follow those of matrix i - 1 in the grid, and a workgroup
// finds its matrix by comparing its index with the running tile counts.  A launch of 17.8 or 45.8 MB is paced by its ramp and its
// tail, not by bandwidth; two or three of them in one launch are one ramp and one tail.  count == 0: the kernel's own arguments
// describe the one matrix.
constexpr int BQ_MULTI_MAX = 8;
struct BqMulti
{
    int count;
    int tile_end[BQ_MULTI_MAX]; // first tile (of the whole launch) that no longer belongs to matrix i
    int N[BQ_MULTI_MAX];
    int bt[BQ_MULTI_MAX];
    float alpha[BQ_MULTI_MAX], beta[BQ_MULTI_MAX];
    const unsigned char* wpk[BQ_MULTI_MAX];
    const float4* dpk[BQ_MULTI_MAX];
    const float* c[BQ_MULTI_MAX];
    float* out[BQ_MULTI_MAX];
    size_t out_stride[BQ_MULTI_MAX];
};

// the halves layout (see blockquant8_upfront_kernel): everything but 8-bit fields in blocks of 64 or 128
static inline bool halves_layout(int bits, int block)
{
    return bits != 8 || block == 32;
}

// Many rows of fp16 activations (blockquant_rows.hip; many_rows_f16 in blockquant.hip says from how many: 17 always, 5 on large
// weights): every matrix of mm on the same rows, one launch.
int launch_blockquant_rows_f16(const uint16_t* a, size_t a_stride, int M, int K, int bits, int block, const BqMulti& mm, hipStream_t stream);

// The same with fp32 rows (16-byte aligned) and optional input scales; and about how long that takes for `count` matrices of N[i] rows, with the shape
// it will take.
double blockquant_rows_f32_us(int M, int K, const int* N, int count, int* mg, int* rt);
int launch_blockquant_rows_f32(const float* a, size_t a_stride, int M, int K, int bits, int block, const float* in_scales, const BqMulti& mm, hipStream_t stream);

// Many rows of fp32 activations, weights in blocks of 64 or 128 (blockquant_tiles.hip); the workspace is that of ncnnhip_gemm_blockquant_packed_rows.
int launch_blockquant_tiles(const float* a, size_t a_stride, int M, int N, int K, int bits, const unsigned char* wpk, const float4* dpk, const float* in_scales,
                            const float* c, int bt, float alpha, float beta, float* out, size_t out_stride, void* workspace, hipStream_t stream);

} // namespace ncnnhip

#endif // NCNNHIP_BLOCKQUANT_H
