// The attention core of MultiHeadAttention (src/layer/multiheadattention.cpp:776-866 in the block-quantised forward):
// per head  out = softmax(q k^T + mask) v  in fp32.  The four projections around it are block-quantised Gemms.
//
// Layouts: q and out are [sequence][embed_dim] (row = token); keys and values are [embed_dim][dst_seqlen], one row per
// channel over time, which is the layout the reference layer hands out and takes back as its cache.
//
// One workgroup = up to 4 query rows of one head.
//   scores : thread j owns key j, walks the head's channels in order (the reference's summation order, no FMA) reading
//            k[channel][j] coalesced; the 4 queries reuse every key value loaded
//   softmax: one wavefront per query row (max, exp, sum by shuffles), probabilities stay in LDS
//   p v    : a wavefront takes channels w, w+4, ...; lanes stride over time reading v[channel][k] coalesced, then a
//            shuffle reduction (so the sum over k is a tree, not the reference's sequence: fp32 tolerance)
#include <float.h>
#include <limits.h>

#include "common.h"

namespace ncnnhip {

static constexpr int ATT_TQ = 4;

__device__ __forceinline__ float wave_max(float v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}
__device__ __forceinline__ float wave_sum(float v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = add_rn(v, __shfl_xor(v, o));
    return v;
}

__global__ __launch_bounds__(256) void attention_f32_kernel(const float* __restrict__ q, const float* __restrict__ kt, const float* __restrict__ vt,
                                                            const float* __restrict__ mask, int mask_heads, int head_dim, int embed_dim, int src, int dst,
                                                            size_t kv_stride, float* __restrict__ out, size_t q_stride, float q_scale)
{
    extern __shared__ float smem[];
    float* qs = smem;                     // [ATT_TQ][head_dim]
    float* sc = smem + ATT_TQ * head_dim; // [ATT_TQ][dst]
    const int h = blockIdx.y;
    const int i0 = blockIdx.x * ATT_TQ;
    const int rows = src - i0 < ATT_TQ ? src - i0 : ATT_TQ;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

    for (int e = tid; e < ATT_TQ * head_dim; e += 256)
    {
        const int t = e / head_dim, l = e - t * head_dim;
        qs[e] = t < rows ? mul_rn(q[(size_t)(i0 + t) * q_stride + h * head_dim + l], q_scale) : 0.f;
    }
    __syncthreads();

    // ---- scores
    const float* kh = kt + (size_t)h * head_dim * kv_stride;
    for (int j = tid; j < dst; j += 256)
    {
        float acc[ATT_TQ];
#pragma unroll
        for (int t = 0; t < ATT_TQ; t++) acc[t] = 0.f;
        for (int l = 0; l < head_dim; l++)
        {
            const float kv = kh[(size_t)l * kv_stride + j];
#pragma unroll
            for (int t = 0; t < ATT_TQ; t++) acc[t] = add_rn(acc[t], mul_rn(qs[t * head_dim + l], kv));
        }
#pragma unroll
        for (int t = 0; t < ATT_TQ; t++)
        {
            float s = acc[t];
            if (mask && t < rows) s = add_rn(s, mask[((size_t)(mask_heads > 1 ? h : 0) * src + i0 + t) * dst + j]);
            sc[t * dst + j] = s;
        }
    }
    __syncthreads();

    // ---- softmax, wavefront `wave` owns query row `wave`
    {
        float* row = sc + wave * dst;
        float mx = -FLT_MAX;
        for (int j = lane; j < dst; j += 64) mx = fmaxf(mx, row[j]);
        mx = wave_max(mx);
        float total = 0.f;
        for (int j = lane; j < dst; j += 64)
        {
            const float e = expf(add_rn(row[j], -mx));
            row[j] = e;
            total = add_rn(total, e);
        }
        total = wave_sum(total);
        for (int j = lane; j < dst; j += 64) row[j] = div_rn(row[j], total);
    }
    __syncthreads();

    // ---- probabilities times values
    const float* vh = vt + (size_t)h * head_dim * kv_stride;
    for (int l = wave; l < head_dim; l += 4)
    {
        const float* vr = vh + (size_t)l * kv_stride;
        float acc[ATT_TQ];
#pragma unroll
        for (int t = 0; t < ATT_TQ; t++) acc[t] = 0.f;
        for (int k = lane; k < dst; k += 64)
        {
            const float v = vr[k];
#pragma unroll
            for (int t = 0; t < ATT_TQ; t++) acc[t] = add_rn(acc[t], mul_rn(sc[t * dst + k], v));
        }
#pragma unroll
        for (int t = 0; t < ATT_TQ; t++)
        {
            const float s = wave_sum(acc[t]);
            if (lane == 0 && t < rows) out[(size_t)(i0 + t) * embed_dim + h * head_dim + l] = s;
        }
    }
}

// ---- the same on the fp32 matrix cores, for head dimensions 32 / 64 / 96 / 128 ------------------------------------
// One workgroup = 32 query rows of one head; its 4 wavefronts take key tiles (32 keys) in turn and each keeps a
// running softmax (maximum m, sum l, unnormalised output) for its share; the shares are merged at the end.
// Everything is computed transposed, so that both MFMA operands come straight from where they lie:
//   S^T = K Q^T : A = k[channel][key] read coalesced along the keys, B = q values held in registers.  The result has
//                 keys down the registers and the 32 queries across the lanes: a query's softmax is per-lane arithmetic
//                 plus one exchange with lane^32.
//   O^T = V P^T : B = exp(S^T - m) is used from the accumulator registers as they are: MFMA step kk of half hh is given
//                 key 8*(kk/4) + 4*hh + kk%4, the key that register kk of that lane holds; A = v[channel][key] with the
//                 same key order, four 16-byte loads per lane and 32 channels.
// Scores and products are fp32 throughout; the order of the additions (and the running rescale by exp(m_old - m_new))
// differs from the reference's two-pass softmax: compared with an fp32 tolerance.
// e^x for x <= 0 in three instructions: the hardware's 2^y (1 ulp) on y = x * log2(e).  Rounding y moves the result by at most
// |y| * 2^-24 of itself, so a term of relative size e^x carries an error below 2^-24 * |x| e^x <= 2.2e-8 of the row's largest
// term; -inf and differences beyond the exponent range give 0.  (The library's expf spends 14 instructions on range
// reduction and range checks; with 16 probabilities per lane and tile that was the largest part of the vector work.)
__device__ __forceinline__ float exp_of_nonpositive(float x)
{
    return __builtin_amdgcn_exp2f(mul_rn(x, 1.44269504088896341f));
}

typedef float v16f_at __attribute__((ext_vector_type(16)));
typedef float v4f_at __attribute__((ext_vector_type(4)));

// Nothing moves across it: the empty asm holds memory accesses in place for the passes that work on the IR, the scheduling
// barrier holds every instruction in place for the machine scheduler.
#define ATT_PHASE_BOUNDARY()                \
    do                                      \
    {                                       \
        asm volatile("" ::: "memory");      \
        __builtin_amdgcn_sched_barrier(0);  \
    } while (0)

// the 16 values of one channel that a lane feeds to the products of O^T: keys j0 + 8*(kk/4) + 4*hh + kk%4
__device__ __forceinline__ void load_value_block(float (&vv)[16], const float* __restrict__ vr, int j0, int hh, int dst, bool vec)
{
    if (vec)
    {
#pragma unroll
        for (int a = 0; a < 4; a++)
        {
            const v4f_at t4 = *reinterpret_cast<const v4f_at*>(vr + j0 + 8 * a + 4 * hh);
#pragma unroll
            for (int e = 0; e < 4; e++) vv[4 * a + e] = t4[e];
        }
    }
    else
    {
#pragma unroll
        for (int kk = 0; kk < 16; kk++)
        {
            const int key = j0 + 8 * (kk >> 2) + 4 * hh + (kk & 3);
            vv[kk] = vr[key < dst ? key : dst - 1]; // past the end: its probability is 0
        }
    }
}

// One tile's step of the running softmax of a query (lanes l and l^32 hold the two halves of its 32 scores): scores
// become exp(score - new maximum), the running sum and maximum are brought up to date, and the factor that rescales what
// was accumulated under the old maximum is returned.
__device__ __forceinline__ float running_softmax_step(v16f_at& s, float& m, float& l)
{
    float mx = -FLT_MAX;
#pragma unroll
    for (int r = 0; r < 16; r++) mx = fmaxf(mx, s[r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float m_new = fmaxf(m, mx);
    const float corr = exp_of_nonpositive(m - m_new);
    float psum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; r++)
    {
        s[r] = exp_of_nonpositive(s[r] - m_new);
        psum += s[r];
    }
    psum += __shfl_xor(psum, 32);
    l = l * corr + psum;
    m = m_new;
    return corr;
}

// A wavefront's share of the keys [key_begin, key_end) for the 32 queries of its workgroup: maximum, sum and unnormalised output (transposed)
template<int HD>
__device__ __forceinline__ void attention_share_f32(const float* __restrict__ q, int qi, int h, const float* __restrict__ kt, const float* __restrict__ vt, const float* mrow,
                                                    int dst, size_t kv_stride, int v_vec_ok, int key_begin, int key_end, size_t q_stride, float q_scale,
                                                    v16f_at (&o)[HD / 32], float& m, float& l)
{
    constexpr int CB = HD / 32;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l32 = lane & 31, hh = lane >> 5;
    float qreg[HD / 2];
#pragma unroll
    for (int kk = 0; kk < HD / 2; kk++) qreg[kk] = mul_rn(q[(size_t)qi * q_stride + h * HD + 2 * kk + hh], q_scale);

#pragma unroll
    for (int cb = 0; cb < CB; cb++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[cb][r] = 0.f;
    m = -FLT_MAX;
    l = 0.f;

    const float* kh = kt + (size_t)h * HD * kv_stride;
    const float* vh = vt + (size_t)h * HD * kv_stride;
    // Key loads: channel pair kk starts at a wave-uniform address (scalar registers), the lane adds one 32-bit offset that
    // is the same for every kk (the host checks that kv_stride + dst fits) - 64-bit per-lane addresses for 32 rows would
    // cost 64 registers and with them the second wavefront per SIMD.
    //
    // The loop is pipelined by hand over the wavefront's tiles of 32 keys.  Iteration t:
    //   (1) request the values of tile t (and its mask values), (2) add the mask / drop keys past the end in the scores of
    //   tile t, which the previous iteration left in s_cur, (3) the products of S^T for tile t+1 (its keys were requested
    //   one iteration ago) together with the softmax arithmetic of tile t: one block of code, the vector instructions
    //   issue while the matrix pipe works on the chain of products, (4) request the keys of tile t+2, (5) the products
    //   of O^T for tile t.
    // The phase boundaries keep the compiler from sinking loads back to their first use (left to itself it keeps one to
    // eight loads in flight and a wavefront stands on each latency in turn).
    constexpr int VB = CB <= 2 ? CB : 1; // value blocks requested ahead: all of them while the registers last, else one at a time
    const int j_first = key_begin + wave * 32;
    float kreg[HD / 2];
    v16f_at s_cur;
#pragma unroll
    for (int r = 0; r < 16; r++) s_cur[r] = 0.f;
    if (j_first < key_end)
    {
        {
            const unsigned koff = (unsigned)hh * (unsigned)kv_stride + (unsigned)(j_first + l32 < dst ? j_first + l32 : dst - 1);
#pragma unroll
            for (int kk = 0; kk < HD / 2; kk++) kreg[kk] = (kh + (size_t)(2 * kk) * kv_stride)[koff];
        }
        ATT_PHASE_BOUNDARY();
#pragma unroll
        for (int kk = 0; kk < HD / 2; kk++) s_cur = __builtin_amdgcn_mfma_f32_32x32x2f32(kreg[kk], qreg[kk], s_cur, 0, 0, 0);
        asm volatile("" : "+v"(s_cur)); // the products are pure arithmetic and would be sunk past the boundary to their first use: this pins them before it
        ATT_PHASE_BOUNDARY();
        {
            // past the last tile of this wavefront the loads repeat a key and are never used
            const int jn = j_first + 128 < key_end ? j_first + 128 : j_first;
            const unsigned koff = (unsigned)hh * (unsigned)kv_stride + (unsigned)(jn + l32 < dst ? jn + l32 : dst - 1);
#pragma unroll
            for (int kk = 0; kk < HD / 2; kk++) kreg[kk] = (kh + (size_t)(2 * kk) * kv_stride)[koff];
        }
    }
    for (int j0 = j_first; j0 < key_end; j0 += 128)
    {
        const bool full = j0 + 32 <= dst;
        float vv[VB][16];
        if constexpr (CB <= 2)
        {
#pragma unroll
            for (int cb = 0; cb < CB; cb++) load_value_block(vv[cb], vh + (size_t)(cb * 32 + l32) * kv_stride, j0, hh, dst, full && v_vec_ok);
        }
        // register r of this lane: key j0 + 8*(r/4) + 4*hh + r%4 for query l32
        if (mrow)
        {
            // all 16 mask values requested before the first is used; a key past the end repeats the last one and is dropped below
            float mv[16];
#pragma unroll
            for (int r = 0; r < 16; r++)
            {
                const int key = j0 + 8 * (r >> 2) + 4 * hh + (r & 3);
                mv[r] = mrow[key < dst ? key : dst - 1];
            }
#pragma unroll
            for (int r = 0; r < 16; r++) s_cur[r] = add_rn(s_cur[r], mv[r]);
        }
        if (!full)
        {
#pragma unroll
            for (int r = 0; r < 16; r++)
                if (j0 + 8 * (r >> 2) + 4 * hh + (r & 3) >= dst) s_cur[r] = -INFINITY;
        }
        ATT_PHASE_BOUNDARY();
        v16f_at s_next;
#pragma unroll
        for (int r = 0; r < 16; r++) s_next[r] = 0.f;
        float corr;
        if (j0 + 128 < key_end)
        {
#pragma unroll
            for (int kk = 0; kk < HD / 2; kk++) s_next = __builtin_amdgcn_mfma_f32_32x32x2f32(kreg[kk], qreg[kk], s_next, 0, 0, 0);
            corr = running_softmax_step(s_cur, m, l);
            // issue order within the block: one product, then three of the vector instructions, while these last
#pragma unroll
            for (int kk = 0; kk < HD / 2; kk++)
            {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
            }
        }
        else
            corr = running_softmax_step(s_cur, m, l);
        asm volatile("" : "+v"(s_next), "+v"(s_cur));
        ATT_PHASE_BOUNDARY();
        {
            const int jn = j0 + 256 < key_end ? j0 + 256 : j0;
            const unsigned koff = (unsigned)hh * (unsigned)kv_stride + (unsigned)(jn + l32 < dst ? jn + l32 : dst - 1);
#pragma unroll
            for (int kk = 0; kk < HD / 2; kk++) kreg[kk] = (kh + (size_t)(2 * kk) * kv_stride)[koff];
        }
        ATT_PHASE_BOUNDARY();
#pragma unroll
        for (int cb = 0; cb < CB; cb++)
        {
#pragma unroll
            for (int r = 0; r < 16; r++) o[cb][r] *= corr;
            if constexpr (CB > 2) load_value_block(vv[0], vh + (size_t)(cb * 32 + l32) * kv_stride, j0, hh, dst, full && v_vec_ok);
#pragma unroll
            for (int kk = 0; kk < 16; kk++) o[cb] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv[CB <= 2 ? cb : 0][kk], s_cur[kk], o[cb], 0, 0, 0);
        }
        s_cur = s_next;
    }
}

// The four wavefronts' shares become the result, or the record of a key split
template<int HD>
__device__ __forceinline__ void attention_merge_shares(const v16f_at (&o)[HD / 32], float m, float l, int h, int i0, int src, int embed_dim, float* __restrict__ out,
                                                       bool split, float* __restrict__ rec)
{
    constexpr int CB = HD / 32;
    constexpr int LD = 33;
    __shared__ float o_s[HD * LD];
    __shared__ float m_s[4][32], l_s[4][32];
    unsigned thread = threadIdx.x;
    // Head dimension 96 has no register to spare: with what is made of the thread's number kept from before the loop it took 257 and one wavefront ran
    // on a SIMD instead of two.  (us, 257 registers and 255: fp32 core, 27 heads, 28 queries on 1504 keys 44.3 38.0; split core, 22 heads, 1710 on
    // 1731 284 210, 15 heads, 1862 on 3740 436 287.  The others have registers enough and are 2 to 4 % slower this way on short sequences.)
    if constexpr (HD == 96) asm volatile("" : "+v"(thread));
    const int tid = (int)thread, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, hh = lane >> 5;
    if (hh == 0)
    {
        m_s[wave][l32] = m;
        l_s[wave][l32] = l;
    }
    __syncthreads();
    const float mall = fmaxf(fmaxf(m_s[0][l32], m_s[1][l32]), fmaxf(m_s[2][l32], m_s[3][l32]));
    const float f = expf(m - mall); // a wavefront that saw no key has m = -FLT_MAX, l = 0, o = 0
    for (int w = 0; w < 4; w++)
    {
        if (wave == w)
        {
#pragma unroll
            for (int cb = 0; cb < CB; cb++)
#pragma unroll
                for (int r = 0; r < 16; r++)
                {
                    const int ch = cb * 32 + 8 * (r >> 2) + 4 * hh + (r & 3);
                    const float v = o[cb][r] * f;
                    o_s[ch * LD + l32] = w == 0 ? v : o_s[ch * LD + l32] + v;
                }
        }
        __syncthreads();
    }
    if (split)
    {
        // a record: 32 maxima, 32 sums, 32 x HD outputs (query-major; only real queries are written)
        const int nq = src - i0 < 32 ? src - i0 : 32;
        if (tid < 32)
        {
            const float ma = fmaxf(fmaxf(m_s[0][tid], m_s[1][tid]), fmaxf(m_s[2][tid], m_s[3][tid]));
            float lt = 0.f;
#pragma unroll
            for (int w = 0; w < 4; w++) lt += l_s[w][tid] * expf(m_s[w][tid] - ma);
            rec[tid] = ma;
            rec[32 + tid] = lt;
        }
        for (int idx = tid; idx < nq * HD; idx += 256) rec[64 + idx] = o_s[(idx % HD) * LD + idx / HD];
        return;
    }
    for (int idx = tid; idx < 32 * HD; idx += 256)
    {
        const int qq = idx / HD, ch = idx - qq * HD;
        if (i0 + qq < src)
        {
            float lt = 0.f;
#pragma unroll
            for (int w = 0; w < 4; w++) lt += l_s[w][qq] * expf(m_s[w][qq] - fmaxf(fmaxf(m_s[0][qq], m_s[1][qq]), fmaxf(m_s[2][qq], m_s[3][qq])));
            out[(size_t)(i0 + qq) * embed_dim + h * HD + ch] = div_rn(o_s[ch * LD + qq], lt);
        }
    }
}

template<int HD>
__global__ __launch_bounds__(256) void attention_f32_mfma_kernel(const float* __restrict__ q, const float* __restrict__ kt, const float* __restrict__ vt,
                                                                 const float* __restrict__ mask, int mask_heads, int embed_dim, int src, int dst,
                                                                 size_t kv_stride, float* __restrict__ out, int v_vec_ok, int keys_per_split,
                                                                 float* __restrict__ partial, size_t q_stride, float q_scale)
{
    // keys_per_split > 0: blockIdx.z takes keys [z*keys_per_split, ...) and leaves (m, l, unnormalised o) in `partial`
    // for attention_merge_kernel; 0: the workgroup sees every key and writes the result
    const int h = blockIdx.y, i0 = blockIdx.x * 32, l32 = threadIdx.x & 31;
    const int qi = i0 + l32 < src ? i0 + l32 : src - 1; // lanes past the last query repeat it; nothing of theirs is stored
    const float* mrow = mask ? mask + ((size_t)(mask_heads > 1 ? h : 0) * src + qi) * dst : nullptr;
    const int key_begin = keys_per_split > 0 ? (int)blockIdx.z * keys_per_split : 0;
    const int key_end = keys_per_split > 0 && key_begin + keys_per_split < dst ? key_begin + keys_per_split : dst; // a multiple of 32, or dst
    v16f_at o[HD / 32];
    float m, l;
    attention_share_f32<HD>(q, qi, h, kt, vt, mrow, dst, kv_stride, v_vec_ok, key_begin, key_end, q_stride, q_scale, o, m, l);
    // records: [head][query block][split]
    attention_merge_shares<HD>(o, m, l, h, i0, src, embed_dim, out, keys_per_split > 0,
                               partial + (((size_t)h * gridDim.x + blockIdx.x) * gridDim.z + blockIdx.z) * (size_t)(64 + HD * 32));
}

// ---- the same on the bf16 matrix cores, every fp32 number as three bf16 numbers ----------------------------------------
// x = hi + mid + lo, each the nearest bf16 of what is left: 24 bits, exact, the remainders of either sign.  A product is then the six
// products hi hi, hi mid, mid hi, mid mid, hi lo, lo hi; what is left out, mid lo, lo mid and lo lo, is at most 2^-23 of it, of random
// sign.  Six instructions of 32 x 32 x 16 in place of eight of 32 x 32 x 2 at a sixteenth of the rate: 1536 matrix-core cycles for 32 keys
// and queries at head dimension 64 where the kernel above takes 4096.  The least products are added first.
// Keys and values are split once, by attention_split_kernel, into the workspace, in operand order: per head and 32 keys the HD / 16 x 3
// fragments of the keys and the HD / 16 x 3 of the values, 64 lanes x 16 bytes each, so that every load of the core is 1 KB of consecutive
// memory.  The queries' fragments are made by the workgroup and stay in LDS (in registers, 96 of them at head dimension 64, short sequences
// run 5 % longer and the longest 2 % shorter).
// Bound by the matrix cores and the vector unit (softmax, the probabilities' split) of two wavefronts per SIMD: at head dimension 64 an
// iteration is 1536 cycles of products and takes 4500 for two wavefronts.  16 heads of 64: 1500 queries and keys 134 us -> 82 with
// attention_split_kernel and the merge, 700: 57 -> 34; 12 of 128, 500: 83 -> 35; 20 of 96, 300 on 600: 75 -> 34.
// (Three wavefronts per SIMD in 168 registers, eight to a workgroup, or a start at another key for each workgroup: no faster.)
// An infinity times a part that is zero is no number where the product of the whole was one; a wavefront that ends with one repeats its
// share with the kernel above's arithmetic.  So that it does, eight numbers of a key, value or query among which one is below 2^-110, where
// bf16 has no bits for the least part, are stored as no numbers (left as they are, values of 2^-116 gave a relative error of 2.3e-6 and of
// 2^-122 1.4e-4).  A probability below 2^-117, whose exponential is 2^-19 off at best, keeps what lies above 2^-134.
typedef __bf16 v8bf_at __attribute__((ext_vector_type(8)));

// two floats -> their three bf16 pairs; returns whether anything is left
__device__ __forceinline__ unsigned split_pair(float a, float b, unsigned (&part)[3])
{
#pragma unroll
    for (int p = 0; p < 3; p++)
    {
        asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(part[p]) : "v"(a), "v"(b));
        a -= __uint_as_float(part[p] << 16);
        b -= __uint_as_float(part[p] & 0xFFFF0000u);
    }
    return __float_as_uint(a) | __float_as_uint(b);
}
__device__ __forceinline__ void split_store(const float (&x)[8], uint4* to, int stride) // to, to + stride, to + 2 * stride
{
    unsigned f[4][3], left = 0;
#pragma unroll
    for (int e = 0; e < 4; e++) left |= split_pair(x[2 * e], x[2 * e + 1], f[e]);
    f[0][0] = left ? 0x7FC07FC0u : f[0][0]; // no number: see above
#pragma unroll
    for (int p = 0; p < 3; p++) to[p * stride] = make_uint4(f[0][p], f[1][p], f[2][p], f[3][p]);
}

// One workgroup: 32 keys of one head.  new_k / new_v (or null): the keys and values of the positions from `past` on, rows of new_stride floats
// ([position][embed]); they are copied into kt / vt on the way (appending to the cache is then no launch of its own).
// Bound by memory, with 20 bytes moved for a float (28 for a new one), and on few keys by its latency: every load of a thread is requested
// before the first is used, and LDS is sized by the head dimension (1500 new keys of 16 heads of 64, 43 MB: 13 us with loads as they come
// and room for 128 channels in 32 KB).
template<int HD>
__global__ __launch_bounds__(256) void attention_split_kernel(float* kt, float* vt, size_t kv_stride, int dst, const float* __restrict__ new_k,
                                                              const float* __restrict__ new_v, size_t new_stride, int past, uint4* __restrict__ frags)
{
    constexpr int EACH = HD / 8, STEPS = HD / 16;
    __shared__ float tile[2][HD][33];
    const int j0 = blockIdx.x * 32, h = blockIdx.y, tid = threadIdx.x;
    const size_t row0 = (size_t)h * HD;
    const int known = new_k ? past : dst; // columns of kt / vt that are there
    float x[2][EACH];
    // channel-major from kt / vt, thread = (key, every eighth channel); position-major from the new rows, consecutive threads = consecutive channels
    const int key = tid & 31, c0 = tid >> 5, j = j0 + key;
    if (j0 < known || j0 + 32 > dst) // uniform, like the next: a tile may be of both kinds
    {
        const size_t at = (row0 + c0) * kv_stride + j;
        const bool there = j < known;
#pragma unroll
        for (int i = 0; i < EACH; i++)
        {
            x[0][i] = there ? kt[at + (size_t)(8 * i) * kv_stride] : 0.f;
            x[1][i] = there ? vt[at + (size_t)(8 * i) * kv_stride] : 0.f;
        }
        if (there || j >= dst)
        {
#pragma unroll
            for (int i = 0; i < EACH; i++)
            {
                tile[0][c0 + 8 * i][key] = x[0][i];
                tile[1][c0 + 8 * i][key] = x[1][i];
            }
        }
    }
    if (j0 + 32 > known)
    {
#pragma unroll
        for (int i = 0; i < EACH; i++)
        {
            const int e = tid + 256 * i, k = e / HD, c = e - k * HD, jn = j0 + k;
            const bool fresh = jn >= known && jn < dst;
            const size_t from = (size_t)(fresh ? jn - past : 0) * new_stride + row0 + c;
            x[0][i] = new_k ? new_k[from] : 0.f;
            x[1][i] = new_k ? new_v[from] : 0.f;
        }
#pragma unroll
        for (int i = 0; i < EACH; i++)
        {
            const int e = tid + 256 * i, k = e / HD, c = e - k * HD, jn = j0 + k;
            if (jn >= known && jn < dst)
            {
                tile[0][c][k] = x[0][i];
                tile[1][c][k] = x[1][i];
            }
        }
    }
    __syncthreads();
    if (j >= known && j < dst)
    {
#pragma unroll
        for (int i = 0; i < EACH; i++)
        {
            kt[(row0 + c0 + 8 * i) * kv_stride + j] = tile[0][c0 + 8 * i][key];
            vt[(row0 + c0 + 8 * i) * kv_stride + j] = tile[1][c0 + 8 * i][key];
        }
    }
    uint4* to = frags + ((size_t)h * gridDim.x + blockIdx.x) * (size_t)(STEPS * 6 * 64);
    for (int e = tid; e < STEPS * 64; e += 256)
    {
        const int step = e >> 6, lane = e & 63, l32 = lane & 31, hh = lane >> 5;
        float y[8];
        // keys: lane = key, channels step * 16 + hh * 8 ..; values: step = 32 channels and half of the keys, in the order of the accumulators
#pragma unroll
        for (int i = 0; i < 8; i++) y[i] = tile[0][step * 16 + hh * 8 + i][l32];
        split_store(y, to + step * 3 * 64 + lane, 64);
#pragma unroll
        for (int i = 0; i < 8; i++) y[i] = tile[1][(step >> 1) * 32 + l32][(step & 1) * 16 + 8 * (i >> 2) + 4 * hh + (i & 3)];
        split_store(y, to + (STEPS + step) * 3 * 64 + lane, 64);
    }
}

template<int HD>
__global__ __launch_bounds__(256, HD <= 64 ? 2 : 1) void attention_bf16x3_kernel(const float* __restrict__ q, const float* __restrict__ kt, const float* __restrict__ vt,
                                                               const uint4* __restrict__ frags, const float* __restrict__ mask, int mask_heads, int embed_dim, int src,
                                                               int dst, size_t kv_stride, float* __restrict__ out, int v_vec_ok, int keys_per_split,
                                                               float* __restrict__ partial, size_t q_stride, float q_scale, int query_blocks, int splits)
{
    constexpr int CB = HD / 32, STEPS = HD / 16;
    __shared__ uint4 q_s[STEPS * 3 * 64];
    // The query blocks of a head read the same fragments, 384 bytes a key and 32 channels: they follow one another on one die (workgroups are
    // dealt to the 8 dies in turn), whose L2 then holds a few heads at a time instead of all of them (16 heads of 64, 256 queries, 2304 keys:
    // 64 us without, 46 with).  With `splits` beyond 1 that many workgroups share a unit's keys.
    const int T = gridDim.x, die = blockIdx.x & 7, more = T & 7, at = die * (T >> 3) + (die < more ? die : more) + (int)(blockIdx.x >> 3);
    const int unit = at / splits, z = at - unit * splits;
    const int h = unit / query_blocks, i0 = (unit - h * query_blocks) * 32;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, hh = lane >> 5;
    const int qi = i0 + l32 < src ? i0 + l32 : src - 1; // lanes past the last query repeat it; nothing of theirs is stored
    const float* mrow = mask ? mask + ((size_t)(mask_heads > 1 ? h : 0) * src + qi) * dst : nullptr;
    const int key_begin = z * keys_per_split;
    const int key_end = splits > 1 && key_begin + keys_per_split < dst ? key_begin + keys_per_split : dst; // a multiple of 32, or dst

    for (int step = wave; step < STEPS; step += 4)
    {
        const float* from = q + (size_t)qi * q_stride + h * HD + step * 16 + hh * 8;
        float x[8];
#pragma unroll
        for (int i = 0; i < 8; i++) x[i] = mul_rn(from[i], q_scale);
        split_store(x, q_s + step * 3 * 64 + lane, 64);
    }
    __syncthreads();

    union Frag
    {
        uint4 u;
        v8bf_at h;
    };
    v16f_at o[CB];
#pragma unroll
    for (int cb = 0; cb < CB; cb++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[cb][r] = 0.f;
    float m = -FLT_MAX, l = 0.f;
    // pairs (of the first operand, of the second) in the order they are added
    constexpr int PA[6] = {1, 0, 2, 0, 1, 0}, PB[6] = {1, 2, 0, 1, 0, 0};

    const int t_first = key_begin / 32 + wave, t_end = (key_end + 31) / 32;
    const uint4* base = frags + (size_t)h * ((dst + 31) / 32) * (size_t)(STEPS * 6 * 64) + lane;
    Frag kf[STEPS * 3];
    auto load_keys = [&](int t) {
        const uint4* f = base + (size_t)t * (STEPS * 6 * 64);
#pragma unroll
        for (int i = 0; i < STEPS * 3; i++) kf[i].u = f[i * 64];
    };
    auto scores = [&](v16f_at& s) {
        unsigned at = lane; // (opaque: the queries' fragments are read again for every tile, not kept in 48 registers)
        asm volatile("" : "+v"(at));
#pragma unroll
        for (int pr = 0; pr < 6; pr++)
#pragma unroll
            for (int step = 0; step < STEPS; step++)
            {
                Frag qf;
                qf.u = q_s[(step * 3 + PB[pr]) * 64 + at];
                s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[step * 3 + PA[pr]].h, qf.h, s, 0, 0, 0);
            }
    };
    v16f_at s_cur;
#pragma unroll
    for (int r = 0; r < 16; r++) s_cur[r] = 0.f;
    // pipelined like the kernel above: the scores of the next tile are made while the softmax of this one runs, its keys are requested an
    // iteration ahead
    if (t_first < t_end)
    {
        load_keys(t_first);
        scores(s_cur);
        asm volatile("" : "+v"(s_cur));
        ATT_PHASE_BOUNDARY();
        load_keys(t_first + 4 < t_end ? t_first + 4 : t_first);
    }
    for (int t = t_first; t < t_end; t += 4)
    {
        const int j0 = t * 32;
        const uint4* vfrom = base + (size_t)t * (STEPS * 6 * 64) + STEPS * 3 * 64;
        constexpr int VB = CB <= 2 ? CB : 1; // value blocks requested ahead: all of them while the registers last, else one at a time
        Frag vf[VB * 6];
        if constexpr (CB <= 2)
        {
#pragma unroll
            for (int i = 0; i < VB * 6; i++) vf[i].u = vfrom[i * 64];
        }
        if (mrow)
        {
            float mv[16];
#pragma unroll
            for (int r = 0; r < 16; r++)
            {
                const int key = j0 + 8 * (r >> 2) + 4 * hh + (r & 3);
                mv[r] = mrow[key < dst ? key : dst - 1];
            }
#pragma unroll
            for (int r = 0; r < 16; r++) s_cur[r] = add_rn(s_cur[r], mv[r]);
        }
        if (j0 + 32 > dst)
        {
#pragma unroll
            for (int r = 0; r < 16; r++)
                if (j0 + 8 * (r >> 2) + 4 * hh + (r & 3) >= dst) s_cur[r] = -INFINITY;
        }
        ATT_PHASE_BOUNDARY();
        v16f_at s_next;
#pragma unroll
        for (int r = 0; r < 16; r++) s_next[r] = 0.f;
        float corr;
        if (t + 4 < t_end)
        {
            scores(s_next);
            corr = running_softmax_step(s_cur, m, l);
            // issue order: one product, then five of the vector instructions, while these last
#pragma unroll
            for (int i = 0; i < STEPS * 6; i++)
            {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 20 / STEPS, 0);
            }
        }
        else
            corr = running_softmax_step(s_cur, m, l);
        asm volatile("" : "+v"(s_next), "+v"(s_cur));
        ATT_PHASE_BOUNDARY();
        load_keys(t + 8 < t_end ? t + 8 : t);
        ATT_PHASE_BOUNDARY();
        if (__any(corr != 1.f))
        {
#pragma unroll
            for (int cb = 0; cb < CB; cb++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[cb][r] *= corr;
        }
        // the probabilities' parts: registers 8 * s .. + 7 are the second operand of the values' step s
        Frag pf[2][3];
#pragma unroll
        for (int s = 0; s < 2; s++)
        {
            unsigned f[4][3];
#pragma unroll
            for (int e = 0; e < 4; e++) split_pair(s_cur[8 * s + 2 * e], s_cur[8 * s + 2 * e + 1], f[e]);
#pragma unroll
            for (int p = 0; p < 3; p++) pf[s][p].u = make_uint4(f[0][p], f[1][p], f[2][p], f[3][p]);
        }
#pragma unroll
        for (int c0 = 0; c0 < CB; c0 += VB)
        {
            if constexpr (CB > 2)
            {
#pragma unroll
                for (int i = 0; i < 6; i++) vf[i].u = vfrom[(c0 * 6 + i) * 64];
            }
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int pr = 0; pr < 6; pr++)
#pragma unroll
                    for (int c = 0; c < VB; c++)
                        o[c0 + c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[c * 6 + s * 3 + PA[pr]].h, pf[s][PB[pr]].h, o[c0 + c], 0, 0, 0);
        }
        s_cur = s_next;
    }
    float nan = l != l ? 1.f : 0.f;
#pragma unroll
    for (int cb = 0; cb < CB; cb++)
#pragma unroll
        for (int r = 0; r < 16; r++) nan = o[cb][r] != o[cb][r] ? 1.f : nan;
    if (__any(nan != 0.f))
        attention_share_f32<HD>(q, qi, h, kt, vt, mrow, dst, kv_stride, v_vec_ok, key_begin, key_end, q_stride, q_scale, o, m, l);
    attention_merge_shares<HD>(o, m, l, h, i0, src, embed_dim, out, splits > 1, partial + ((size_t)unit * splits + z) * (size_t)(64 + HD * 32));
}

// merges the records of the key splits: one workgroup per (head, query block).  First every (split, query) pair gets its factor
// exp(m_split - m) and the queries their sums, through LDS; then the outputs are added with eight independent loads in
// flight per thread (a thread that walks the splits for each of its outputs, one dependent load after the other, took 35 us
// for 64 queries x 16 heads x 11 splits).
__global__ __launch_bounds__(256) void attention_merge_kernel(const float* __restrict__ partial, int query_blocks, int splits, int head_dim,
                                                              int embed_dim, int src, float* __restrict__ out)
{
    __shared__ float fac[64][32]; // splits <= 64 (attention_key_splits)
    __shared__ float l_all[32];
    const int unit = blockIdx.x, h = unit / query_blocks, i0 = (unit - h * query_blocks) * 32;
    const size_t rec_size = (size_t)(64 + head_dim * 32);
    const float* rec0 = partial + (size_t)blockIdx.x * splits * rec_size;
    const int nq = src - i0 < 32 ? src - i0 : 32;
    const int tid = threadIdx.x;
    for (int e = tid; e < splits * 32; e += 256) fac[e >> 5][e & 31] = rec0[(size_t)(e >> 5) * rec_size + (e & 31)];
    __syncthreads();
    if (tid < 32)
    {
        float ma = -FLT_MAX;
        for (int z = 0; z < splits; z++) ma = fmaxf(ma, fac[z][tid]);
        float lt = 0.f;
        for (int z = 0; z < splits; z++)
        {
            const float f = exp_of_nonpositive(fac[z][tid] - ma);
            fac[z][tid] = f;
            lt += rec0[(size_t)z * rec_size + 32 + tid] * f; // independent loads: the compiler keeps several in flight
        }
        l_all[tid] = lt;
    }
    __syncthreads();
    // the outputs of the block are shared out over gridDim.y workgroups (each makes the factors for itself: they are cheap)
    const int total = nq * head_dim, share = (total + (int)gridDim.y - 1) / (int)gridDim.y;
    const int begin = (int)blockIdx.y * share, end = begin + share < total ? begin + share : total;
    for (int idx = begin + tid; idx < end; idx += 256)
    {
        const int qq = idx / head_dim, ch = idx - qq * head_dim;
        const float* op = rec0 + 64 + idx;
        float ot = 0.f;
#pragma unroll 8
        for (int z = 0; z < splits; z++) ot += op[(size_t)z * rec_size] * fac[z][qq];
        out[(size_t)(i0 + qq) * embed_dim + h * head_dim + ch] = div_rn(ot, l_all[qq]);
    }
}

// ---- one to four queries on a long key sequence (a decoding step against a cache) ------------------------------------
// With so few queries the work is reading the keys and values once, and the matrix-core kernel above, built around 32
// queries per workgroup, spends its time in a chain of latencies.  Here one workgroup streams 64 keys of one head:
//   scores : thread = (key, quarter of the channels); k[channel][key] is read coalesced along the keys, the four partial
//            dot products of a key are added through LDS;
//   softmax: wavefront t takes query t (maximum, exp, sum over the 64 keys by shuffles);
//   p v    : thread = (channel, quarter of the keys); v[channel][key] is read as 16-byte pieces along the keys, four lanes
//            add their parts by shuffles.
// It leaves (maximum, sum, unnormalised output) per query for attention_fewq_merge_kernel.  fp32 throughout; the order of
// the additions differs from the reference's: fp32 tolerance.
static constexpr int FEWQ_KEYS = 64;
static constexpr int FEWQ_MAX_HEAD_DIM = 256;

// 16 consecutive values of one channel from key j on: 16-byte pieces where the rows allow, else one by one (a key past the
// end repeats the last one; its probability is 0)
__device__ __forceinline__ void load_fewq_values(float (&vv)[16], const float* __restrict__ vr, int j, int dst, bool vec)
{
    if (vec)
    {
#pragma unroll
        for (int a = 0; a < 4; a++)
        {
            const v4f_at t4 = *reinterpret_cast<const v4f_at*>(vr + j + 4 * a);
#pragma unroll
            for (int e = 0; e < 4; e++) vv[4 * a + e] = t4[e];
        }
    }
    else
    {
#pragma unroll
        for (int e = 0; e < 16; e++) vv[e] = vr[j + e < dst ? j + e : dst - 1];
    }
}
// The slots behind the last key of all hold some key's value a second time: zeros instead, as their probability, zero, times an infinity is no number
__device__ __forceinline__ void drop_fewq_values(float (&vv)[16], int j, int dst)
{
#pragma unroll
    for (int e = 0; e < 16; e++) vv[e] = j + e < dst ? vv[e] : 0.f;
}

// new_k / new_v (or null): the keys and values of the last dst - past positions, rows of new_stride floats ([position][embed]).
// The workgroup whose 64 keys reach past `past` first copies its share of them into kt / vt (appending to the cache is then
// no launch of its own) and reads them back like the rest after a barrier; nobody else reads those columns.
__global__ __launch_bounds__(256) void attention_fewq_split_kernel(const float* __restrict__ q, size_t q_stride, float q_scale, float* kt, float* vt, size_t kv_stride,
                                                                   const float* __restrict__ mask, int mask_heads, int head_dim, int src, int dst, int v_vec_ok,
                                                                   float* __restrict__ partial, const float* __restrict__ new_k, const float* __restrict__ new_v,
                                                                   size_t new_stride, int past)
{
    __shared__ float qs[ATT_TQ * FEWQ_MAX_HEAD_DIM];
    __shared__ float red[4][ATT_TQ][FEWQ_KEYS];
    __shared__ float sc[ATT_TQ][FEWQ_KEYS];
    const int split = blockIdx.x, h = blockIdx.y, i0 = blockIdx.z * ATT_TQ;
    const int rows = src - i0 < ATT_TQ ? src - i0 : ATT_TQ;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int j0 = split * FEWQ_KEYS;

    if (new_k && j0 + FEWQ_KEYS > past) // uniform
    {
        const int kb = j0 > past ? j0 : past, ke = j0 + FEWQ_KEYS < dst ? j0 + FEWQ_KEYS : dst;
        for (int e = tid; e < (ke - kb) * head_dim; e += 256)
        {
            const int pos = e / head_dim, c = e - pos * head_dim;
            const size_t from = (size_t)(kb + pos - past) * new_stride + (size_t)h * head_dim + c;
            const size_t to = ((size_t)h * head_dim + c) * kv_stride + kb + pos;
            kt[to] = new_k[from];
            vt[to] = new_v[from];
        }
        __threadfence_block();
        __syncthreads();
    }
    // every load that does not depend on the scores is requested before the first wait: the first 16 channels of this
    // wavefront's keys, this thread's values of the first 64 channels, the queries
    const int per = (head_dim + 3) >> 2, c0 = wave * per, c1 = c0 + per < head_dim ? c0 + per : head_dim;
    const int key = j0 + lane < dst ? j0 + lane : dst - 1; // past the end: repeated, dropped below
    const float* kp = kt + ((size_t)h * head_dim + c0) * kv_stride + key;
    float kfirst[16];
#pragma unroll
    for (int i = 0; i < 16; i++) kfirst[i] = c0 + i < c1 ? kp[(size_t)i * kv_stride] : 0.f;
    const int kq = tid & 3;
    const bool vec = v_vec_ok && j0 + FEWQ_KEYS <= dst;
    float vfirst[16];
    load_fewq_values(vfirst, vt + ((size_t)h * head_dim + ((tid >> 2) < head_dim ? (tid >> 2) : 0)) * kv_stride, j0 + 16 * kq, dst, vec);
    for (int e = tid; e < ATT_TQ * head_dim; e += 256)
    {
        const int t = e / head_dim, l = e - t * head_dim;
        qs[e] = t < rows ? mul_rn(q[(size_t)(i0 + t) * q_stride + h * head_dim + l], q_scale) : 0.f;
    }
    __syncthreads();

    // ---- scores: wavefront g takes the g-th quarter of the channels, lane = key
    {
        float acc[ATT_TQ];
#pragma unroll
        for (int t = 0; t < ATT_TQ; t++) acc[t] = 0.f;
#pragma unroll
        for (int i = 0; i < 16; i++)
            if (c0 + i < c1)
            {
#pragma unroll
                for (int t = 0; t < ATT_TQ; t++) acc[t] = add_rn(acc[t], mul_rn(qs[t * head_dim + c0 + i], kfirst[i]));
            }
        kp += (size_t)16 * kv_stride;
#pragma unroll 8
        for (int c = c0 + 16; c < c1; c++)
        {
            const float kv = *kp;
            kp += kv_stride;
#pragma unroll
            for (int t = 0; t < ATT_TQ; t++) acc[t] = add_rn(acc[t], mul_rn(qs[t * head_dim + c], kv));
        }
#pragma unroll
        for (int t = 0; t < ATT_TQ; t++) red[wave][t][lane] = acc[t];
    }
    __syncthreads();

    // ---- softmax over this workgroup's keys: wavefront t = query t
    float m_t = -FLT_MAX, l_t = 0.f;
    {
        const int t = wave;
        float s = add_rn(add_rn(red[0][t][lane], red[1][t][lane]), add_rn(red[2][t][lane], red[3][t][lane]));
        const bool live = j0 + lane < dst && t < rows;
        if (live && mask) s = add_rn(s, mask[((size_t)(mask_heads > 1 ? h : 0) * src + i0 + t) * dst + j0 + lane]);
        if (!live) s = -INFINITY;
        m_t = fmaxf(wave_max(s), -FLT_MAX); // a query that is not there (or all keys at -inf): every probability 0
        const float pr = exp_of_nonpositive(s - m_t);
        l_t = wave_sum(pr);
        sc[t][lane] = pr;
    }
    __syncthreads();

    // ---- p v: thread = (channel tid/4, keys 16*(tid%4)..+15), four lanes share a channel
    float* rec = partial + (((size_t)blockIdx.z * gridDim.y + h) * gridDim.x + split) * (size_t)(2 * ATT_TQ + ATT_TQ * head_dim);
    for (int ch = tid >> 2; ch < ((head_dim + 63) & ~63); ch += 64)
    {
        float acc[ATT_TQ];
#pragma unroll
        for (int t = 0; t < ATT_TQ; t++) acc[t] = 0.f;
        if (ch < head_dim)
        {
            float vv[16];
            if (ch < 64)
            {
#pragma unroll
                for (int e = 0; e < 16; e++) vv[e] = vfirst[e];
            }
            else
                load_fewq_values(vv, vt + ((size_t)h * head_dim + ch) * kv_stride, j0 + 16 * kq, dst, vec);
            if (j0 + FEWQ_KEYS > dst) drop_fewq_values(vv, j0 + 16 * kq, dst);
#pragma unroll
            for (int e = 0; e < 16; e++)
#pragma unroll
                for (int t = 0; t < ATT_TQ; t++) acc[t] = add_rn(acc[t], mul_rn(sc[t][16 * kq + e], vv[e]));
        }
#pragma unroll
        for (int t = 0; t < ATT_TQ; t++)
        {
            acc[t] = add_rn(acc[t], __shfl_xor(acc[t], 1));
            acc[t] = add_rn(acc[t], __shfl_xor(acc[t], 2));
        }
        if (kq == 0 && ch < head_dim)
#pragma unroll
            for (int t = 0; t < ATT_TQ; t++) rec[2 * ATT_TQ + t * head_dim + ch] = acc[t];
    }
    if (lane == 0)
    {
        rec[wave] = m_t;
        rec[ATT_TQ + wave] = l_t;
    }
}

// The same for the head dimensions of the matrix-core kernels and TQ queries (the arithmetic of both is the same to the bit): every key and
// value the workgroup needs, 64 x 128 of each at head dimension 128, is requested before the first wait, where the kernel above, which
// has registers for 16 channels and 64, goes to memory four times in a row; and no more queries are multiplied than there are (all four
// cost as long as the loads).  Keys and values past `past` are read where they come from, so that nobody waits for them to be stored.
// Bound by the memory's latency and its rate: 32 heads of 128, one query on 1500 keys (49 MB), with the
// merge, 19.4 -> 14.3 us (16.9 with the pieces of a head on all dies); four queries 32.2 -> 19.8; 16 of 64, one on 1001 10.1 -> 8.3.
template<int HD, int TQ>
__global__ __launch_bounds__(256) void attention_fewq_split_hd_kernel(const float* __restrict__ q, size_t q_stride, float q_scale, float* kt, float* vt, size_t kv_stride,
                                                                      const float* __restrict__ mask, int mask_heads, int src, int dst, int v_vec_ok,
                                                                      float* __restrict__ partial, const float* __restrict__ new_k, const float* __restrict__ new_v,
                                                                      size_t new_stride, int past, int splits)
{
    constexpr int PER = HD / 4, NV = (HD + 63) / 64;
    __shared__ float red[4][TQ][FEWQ_KEYS];
    __shared__ float sc[TQ][FEWQ_KEYS];
    // the pieces of a head follow one another on one die (workgroups are dealt to the 8 dies in turn): rows are not whole cache lines, and
    // neighbours share the lines at their ends
    const int T = gridDim.x, die = blockIdx.x & 7, more = T & 7, unit = die * (T >> 3) + (die < more ? die : more) + (int)(blockIdx.x >> 3);
    const int h = unit / splits, split = unit - h * splits;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j0 = split * FEWQ_KEYS, c0 = wave * PER, kq = tid & 3;
    const bool fresh = new_k && j0 + FEWQ_KEYS > past; // uniform: some of these keys are new
    const int last = fresh ? past - 1 : dst - 1; // keys beyond: repeated here, replaced or dropped below

    float kv[PER], vv[NV][16];
    {
        const float* kp = kt + ((size_t)h * HD + c0) * kv_stride + (j0 + lane < last ? j0 + lane : last);
#pragma unroll
        for (int i = 0; i < PER; i++) kv[i] = kp[(size_t)i * kv_stride];
    }
    const bool vec = v_vec_ok && j0 + FEWQ_KEYS <= last + 1;
#pragma unroll
    for (int i = 0; i < NV; i++)
    {
        const int ch = (tid >> 2) + 64 * i < HD ? (tid >> 2) + 64 * i : HD - 1;
        load_fewq_values(vv[i], vt + ((size_t)h * HD + ch) * kv_stride, j0 + 16 * kq, last + 1, vec);
    }
    if (fresh) // dst - past = src positions
    {
#pragma unroll
        for (int t = 0; t < TQ; t++)
        {
            const size_t row = (size_t)(t < src ? t : src - 1) * new_stride + (size_t)h * HD;
            const int at = past + (t < src ? t : src - 1) - j0; // (in this workgroup's keys, or in those of the one before)
            float nk[PER]; // (the same for the whole wavefront)
#pragma unroll
            for (int i = 0; i < PER; i++) nk[i] = new_k[row + c0 + i];
#pragma unroll
            for (int i = 0; i < PER; i++) asm volatile("" : "+s"(nk[i])); // loaded whether the lane takes it or not
#pragma unroll
            for (int i = 0; i < PER; i++) kv[i] = lane == at ? nk[i] : kv[i];
#pragma unroll
            for (int i = 0; i < NV; i++)
            {
                const float v = new_v[row + ((tid >> 2) + 64 * i < HD ? (tid >> 2) + 64 * i : HD - 1)];
#pragma unroll
                for (int e = 0; e < 16; e++) vv[i][e] = 16 * kq + e == at ? v : vv[i][e];
            }
        }
    }
    if (j0 + FEWQ_KEYS > dst) // uniform: the last workgroup of a head
    {
#pragma unroll
        for (int i = 0; i < NV; i++) drop_fewq_values(vv[i], j0 + 16 * kq, dst);
    }

    // ---- scores: wavefront g takes the g-th quarter of the channels, lane = key
    {
        float acc[TQ];
#pragma unroll
        for (int t = 0; t < TQ; t++) acc[t] = 0.f;
#pragma unroll
        for (int t = 0; t < TQ; t++)
        {
            const float* qp = q + (size_t)(t < src ? t : 0) * q_stride + h * HD + c0; // (the same for the whole wavefront)
#pragma unroll
            for (int i = 0; i < PER; i++) acc[t] = add_rn(acc[t], mul_rn(mul_rn(qp[i], q_scale), kv[i]));
        }
#pragma unroll
        for (int t = 0; t < TQ; t++) red[wave][t][lane] = acc[t];
    }
    __syncthreads();

    // ---- softmax over this workgroup's keys: wavefront t = query t
    float m_t = -FLT_MAX, l_t = 0.f;
    if (wave < TQ)
    {
        const int t = wave;
        float s = add_rn(add_rn(red[0][t][lane], red[1][t][lane]), add_rn(red[2][t][lane], red[3][t][lane]));
        const bool live = j0 + lane < dst && t < src;
        if (live && mask) s = add_rn(s, mask[((size_t)(mask_heads > 1 ? h : 0) * src + t) * dst + j0 + lane]);
        if (!live) s = -INFINITY;
        m_t = fmaxf(wave_max(s), -FLT_MAX); // a query that is not there (or all keys at -inf): every probability 0
        const float pr = exp_of_nonpositive(s - m_t);
        l_t = wave_sum(pr);
        sc[t][lane] = pr;
    }
    __syncthreads();

    // ---- p v: thread = (channel tid/4, keys 16*(tid%4)..+15), four lanes share a channel
    float* rec = partial + ((size_t)h * splits + split) * (size_t)(2 * ATT_TQ + ATT_TQ * HD);
#pragma unroll
    for (int i = 0; i < NV; i++)
    {
        const int ch = (tid >> 2) + 64 * i;
        float acc[TQ];
#pragma unroll
        for (int t = 0; t < TQ; t++)
        {
            acc[t] = 0.f;
#pragma unroll
            for (int e = 0; e < 16; e++) acc[t] = add_rn(acc[t], mul_rn(sc[t][16 * kq + e], vv[i][e]));
            acc[t] = add_rn(acc[t], __shfl_xor(acc[t], 1));
            acc[t] = add_rn(acc[t], __shfl_xor(acc[t], 2));
        }
        if (kq == 0 && ch < HD)
#pragma unroll
            for (int t = 0; t < TQ; t++) rec[2 * ATT_TQ + t * HD + ch] = acc[t];
    }
    if (lane == 0)
    {
        rec[wave] = m_t;
        rec[ATT_TQ + wave] = l_t;
    }
    if (fresh) // the new columns into the cache
    {
        const int kb = j0 > past ? j0 : past, ke = j0 + FEWQ_KEYS < dst ? j0 + FEWQ_KEYS : dst;
        for (int e = tid; e < (ke - kb) * HD; e += 256)
        {
            const int pos = e / HD, c = e - pos * HD;
            const size_t from = (size_t)(kb + pos - past) * new_stride + (size_t)h * HD + c;
            const size_t to = ((size_t)h * HD + c) * kv_stride + kb + pos;
            kt[to] = new_k[from];
            vt[to] = new_v[from];
        }
    }
}

// merges the records of attention_fewq_split_kernel: one workgroup per (head, 64 outputs, group of four queries).  The maxima and
// sums of all splits are fetched side by side into LDS (wavefront t = query t) and turned into one factor per split;
// then four groups of 64 threads each add every fourth split's outputs, eight loads in flight, and the groups' parts
// are added through LDS - a thread that walks the splits one load after the other takes 14 us for 24 of them.
static constexpr int FEWQ_MAX_SPLITS = 512; // 8 per lane of a wavefront in the merge

__global__ __launch_bounds__(256) void attention_fewq_merge_kernel(const float* __restrict__ partial, int splits, int head_dim, int embed_dim, int src,
                                                                   float* __restrict__ out)
{
    __shared__ float fac[ATT_TQ][FEWQ_MAX_SPLITS];
    __shared__ float l_all[ATT_TQ];
    __shared__ float part[4][64];
    const int h = blockIdx.x, i0 = blockIdx.y * ATT_TQ;
    const int rows = src - i0 < ATT_TQ ? src - i0 : ATT_TQ;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const size_t rec_size = (size_t)(2 * ATT_TQ + ATT_TQ * head_dim);
    const float* rec0 = partial + ((size_t)blockIdx.y * gridDim.x + h) * splits * rec_size;
    // Everything up to 32 chunks need is requested before the first wait (one trip to memory instead of three): this lane's
    // maxima and sums of chunks lane, lane + 64, ... and, for its output, the parts of this group's first 8 chunks.
    const int idx = blockIdx.z * 64 + lane;
    const float* op = rec0 + 2 * ATT_TQ + idx;
    float ofirst[8], mz[8], lz[8];
    {
#pragma unroll
        for (int k = 0; k < 8; k++) ofirst[k] = idx < rows * head_dim && wave + 4 * k < splits ? op[(size_t)(wave + 4 * k) * rec_size] : 0.f;
#pragma unroll
        for (int k = 0; k < 8; k++)
        {
            const int z = lane + 64 * k; // FEWQ_MAX_SPLITS = 8 * 64
            mz[k] = z < splits ? rec0[z * rec_size + wave] : -FLT_MAX;
            lz[k] = z < splits ? rec0[z * rec_size + ATT_TQ + wave] : 0.f;
        }
    }
    {
        const int t = wave;
        float ma = -FLT_MAX;
#pragma unroll
        for (int k = 0; k < 8; k++) ma = fmaxf(ma, mz[k]);
        ma = wave_max(ma);
        float lt = 0.f;
#pragma unroll
        for (int k = 0; k < 8; k++)
        {
            const int z = lane + 64 * k;
            const float f = exp_of_nonpositive(mz[k] - ma);
            if (z < splits) fac[t][z] = f;
            lt += lz[k] * f;
        }
        lt = wave_sum(lt);
        if (lane == 0) l_all[t] = lt;
    }
    __syncthreads();
    float ot = 0.f;
    if (idx < rows * head_dim)
    {
        const int t = idx / head_dim;
#pragma unroll
        for (int k = 0; k < 8; k++)
            if (wave + 4 * k < splits) ot += ofirst[k] * fac[t][wave + 4 * k];
#pragma unroll 8
        for (int z = wave + 32; z < splits; z += 4) ot += op[z * rec_size] * fac[t][z];
    }
    part[wave][lane] = ot;
    __syncthreads();
    if (wave == 0 && idx < rows * head_dim)
    {
        const int t = idx / head_dim;
        const float sum = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
        out[(size_t)(i0 + t) * embed_dim + h * head_dim + (idx - t * head_dim)] = div_rn(sum, l_all[t]);
    }
}

// the few-query kernels take over where they apply: up to four queries, a key sequence long enough to be worth splitting
static bool attention_fewq_applies(int head_dim, int src, int dst)
{
    return src <= ATT_TQ && dst >= 256 && dst <= FEWQ_KEYS * FEWQ_MAX_SPLITS && head_dim <= FEWQ_MAX_HEAD_DIM;
}
static size_t attention_fewq_workspace_bytes(int num_heads, int head_dim, int src, int dst)
{
    return (size_t)((src + ATT_TQ - 1) / ATT_TQ) * num_heads * ((dst + FEWQ_KEYS - 1) / FEWQ_KEYS) * (size_t)(2 * ATT_TQ + ATT_TQ * head_dim) * sizeof(float);
}

// how many ways to split the keys: enough workgroups for the chip, at least 128 keys (one tile per wavefront) each.
// (With 256 workgroups or more a split does not pay even where the last round over the chip is mostly empty - 47 query
// blocks x 16 heads at head dimension 64 run in 1.47 rounds of 512: split in two, the kernel took 145 us against 136 and
// the merge another 13.)
static int attention_key_splits(int num_heads, int src, int dst)
{
    const long long groups = (long long)((src + 31) / 32) * num_heads;
    if (groups >= 256 || dst < 256) return 1;
    long long want = (512 + groups - 1) / groups;
    const long long most = dst / 128;
    if (want > most) want = most;
    if (want > 64) want = 64;
    return want < 2 ? 1 : (int)want;
}

// Splitting the keys and values first costs a launch and 20 bytes of traffic for each of their floats, which the query blocks have to win back:
// with Q blocks of 32 queries and head dimension D it pays (us, the fp32 kernel and this one)
//   from D Q = 256 on up to 256 D Q keys x heads: 16 heads of 64, 128 queries: 16.1 13.1 alone, 30.9 27.3 on 1000 keys, 49.7 41.7 on 4000;
//   16 x 128, 64 queries on 4000: 70.2 59.4; beyond, 32 x 128, 64 queries on 4000: 99 131;
//   below that up to 64 D Q: 16 x 64, 64 queries: 13.7 12.2 alone, 21.4 18.0 on 250; beyond, on 1000: 21.6 24.8; 32 x 32, 16 queries on 250: 13.9 15.4;
//   and with 8 blocks always: 16 x 64, 320 queries on 4000: 101 65; 32 x 32 the same: 101 72.
// One tile of keys for one small block of queries stays where it is: 16 x 64, 5 queries: 10.5 10.9.
static bool attention_bf16x3_applies(int num_heads, int head_dim, int src, int dst)
{
    if (head_dim % 32 != 0 || head_dim > 128 || src <= ATT_TQ) return false;
    const long long blocks = (src + 31) / 32, width = head_dim * blocks, keys = (long long)num_heads * dst;
    if (blocks * num_heads > 1 << 20) return false; // the grid is one row of workgroups
    if (dst <= 32 && head_dim <= 64) return false;
    return blocks >= 8 || keys <= (width >= 256 ? 256 : 64) * width;
}
// Its workgroups run two to a CU up to head dimension 96, else one (at 96 counted as one: with twice the splits a few hundred keys took 15 % longer,
// some thousands up to 20 % less).  Units (32 queries of a head) that would leave half of these places empty share their keys out over as many
// workgroups as there are places, at least 128 keys each.  (Rounding up as above, or sharing out the last, partly filled of several
// rounds: 768 units at 1500 keys 82 us without, 88 with.)
static int attention_bf16x3_splits(int num_heads, int head_dim, int src, int dst, int& keys_per_split)
{
    const long long units = (long long)((src + 31) / 32) * num_heads;
    long long want = (head_dim <= 64 ? 512 : 256) / units;
    if (want > dst / 128) want = dst / 128;
    if (want > 64) want = 64;
    keys_per_split = 0;
    if (want < 2) return 1;
    keys_per_split = (int)((dst + want - 1) / want + 31) / 32 * 32;
    return (dst + keys_per_split - 1) / keys_per_split;
}
static size_t attention_record_bytes(int head_dim) { return (size_t)(64 + head_dim * 32) * sizeof(float); }
static size_t attention_records_bytes(int num_heads, int head_dim, int src, int dst)
{
    const int splits = attention_key_splits(num_heads, src, dst);
    return splits > 1 ? (size_t)((src + 31) / 32) * num_heads * splits * attention_record_bytes(head_dim) : 0;
}
// split keys and values, and behind them the records of the key splits
static size_t attention_frags_bytes(int num_heads, int head_dim, int dst)
{
    return (size_t)num_heads * ((dst + 31) / 32) * (size_t)head_dim * 384;
}
static size_t attention_bf16x3_bytes(int num_heads, int head_dim, int src, int dst)
{
    int keys_per_split;
    const int splits = attention_bf16x3_splits(num_heads, head_dim, src, dst, keys_per_split);
    return attention_frags_bytes(num_heads, head_dim, dst) + (splits > 1 ? (size_t)((src + 31) / 32) * num_heads * splits * attention_record_bytes(head_dim) : 0);
}

} // namespace ncnnhip

using namespace ncnnhip;

extern "C" {

int ncnnhip_attention_workspace_bytes(int num_heads, int head_dim, int src_seqlen, int dst_seqlen, size_t* workspace_bytes)
{
    NCNNHIP_REQUIRE(num_heads >= 1 && head_dim >= 1 && src_seqlen >= 1 && dst_seqlen >= 1 && workspace_bytes, "ncnnhip_attention_workspace_bytes: bad argument");
    *workspace_bytes = 0;
    if (head_dim % 32 == 0 && head_dim <= 128) *workspace_bytes = attention_records_bytes(num_heads, head_dim, src_seqlen, dst_seqlen);
    if (attention_bf16x3_applies(num_heads, head_dim, src_seqlen, dst_seqlen))
    {
        const size_t need = attention_bf16x3_bytes(num_heads, head_dim, src_seqlen, dst_seqlen);
        if (need > *workspace_bytes) *workspace_bytes = need;
    }
    if (attention_fewq_applies(head_dim, src_seqlen, dst_seqlen))
    {
        const size_t need = attention_fewq_workspace_bytes(num_heads, head_dim, src_seqlen, dst_seqlen);
        if (need > *workspace_bytes) *workspace_bytes = need;
    }
    return NCNNHIP_OK;
}

// append_k / append_v (or null): new rows to be written into columns past.. of kt / vt before they are read
static int attention_dispatch(const float* q_dev, size_t q_stride, float q_scale, float* kt_dev, float* vt_dev, size_t kv_stride, const float* mask_dev, int mask_heads,
                              int num_heads, int head_dim, int src_seqlen, int dst_seqlen, float* out_dev, void* workspace_dev, size_t workspace_bytes, void* stream,
                              const float* append_k, const float* append_v, size_t append_stride, int past);

int ncnnhip_attention_f32(const float* q_dev, const float* kt_dev, const float* vt_dev, size_t kv_stride, const float* mask_dev, int mask_heads,
                          int num_heads, int head_dim, int src_seqlen, int dst_seqlen, float* out_dev, void* workspace_dev, size_t workspace_bytes,
                          void* stream)
{
    return ncnnhip_attention_f32_strided(q_dev, (size_t)num_heads * (size_t)(head_dim > 0 ? head_dim : 0), 1.f, kt_dev, vt_dev, kv_stride, mask_dev, mask_heads, num_heads,
                                         head_dim, src_seqlen, dst_seqlen, out_dev, workspace_dev, workspace_bytes, stream);
}

int ncnnhip_attention_f32_strided(const float* q_dev, size_t q_stride, float q_scale, const float* kt_dev, const float* vt_dev, size_t kv_stride, const float* mask_dev,
                                  int mask_heads, int num_heads, int head_dim, int src_seqlen, int dst_seqlen, float* out_dev, void* workspace_dev,
                                  size_t workspace_bytes, void* stream)
{
    return attention_dispatch(q_dev, q_stride, q_scale, const_cast<float*>(kt_dev), const_cast<float*>(vt_dev), kv_stride, mask_dev, mask_heads, num_heads, head_dim,
                              src_seqlen, dst_seqlen, out_dev, workspace_dev, workspace_bytes, stream, nullptr, nullptr, 0, 0);
}

int ncnnhip_attention_f32_append(const float* qkv_dev, size_t qkv_stride, float q_scale, float* kt_dev, float* vt_dev, size_t kv_stride, int past_seqlen,
                                 const float* mask_dev, int mask_heads, int num_heads, int head_dim, int src_seqlen, float* out_dev, void* workspace_dev,
                                 size_t workspace_bytes, void* stream)
{
    NCNNHIP_REQUIRE(qkv_dev && num_heads >= 1 && head_dim >= 1 && src_seqlen >= 1 && past_seqlen >= 0, "ncnnhip_attention_f32_append: bad argument");
    const size_t e = (size_t)num_heads * (size_t)head_dim;
    NCNNHIP_REQUIRE(qkv_stride >= 3 * e, "ncnnhip_attention_f32_append: rows of q, k and v need a stride of at least 3 * embed_dim");
    NCNNHIP_REQUIRE(past_seqlen <= INT_MAX - src_seqlen, "ncnnhip_attention_f32_append: sequence too long");
    return attention_dispatch(qkv_dev, qkv_stride, q_scale, kt_dev, vt_dev, kv_stride, mask_dev, mask_heads, num_heads, head_dim, src_seqlen, past_seqlen + src_seqlen,
                              out_dev, workspace_dev, workspace_bytes, stream, qkv_dev + e, qkv_dev + 2 * e, qkv_stride, past_seqlen);
}

} // extern "C"

static int attention_dispatch(const float* q_dev, size_t q_stride, float q_scale, float* kt_dev, float* vt_dev, size_t kv_stride, const float* mask_dev, int mask_heads,
                              int num_heads, int head_dim, int src_seqlen, int dst_seqlen, float* out_dev, void* workspace_dev, size_t workspace_bytes, void* stream,
                              const float* append_k, const float* append_v, size_t append_stride, int past)
{
    NCNNHIP_REQUIRE(q_dev && kt_dev && vt_dev && out_dev, "ncnnhip_attention_f32: null pointer");
    NCNNHIP_REQUIRE(num_heads >= 1 && head_dim >= 1 && src_seqlen >= 1 && dst_seqlen >= 1, "ncnnhip_attention_f32: bad shape");
    NCNNHIP_REQUIRE(num_heads <= 65535, "ncnnhip_attention_f32: more than 65535 heads");
    NCNNHIP_REQUIRE(q_stride >= (size_t)num_heads * (size_t)head_dim, "ncnnhip_attention_f32: query row stride below embed_dim");
    NCNNHIP_REQUIRE(kv_stride >= (size_t)dst_seqlen, "ncnnhip_attention_f32: key/value row stride below dst_seqlen");
    NCNNHIP_REQUIRE(kv_stride + (size_t)dst_seqlen < ((size_t)1 << 30), "ncnnhip_attention_f32: key/value row stride beyond the 32-bit byte offsets of the kernel");
    NCNNHIP_REQUIRE(!mask_dev || mask_heads == 1 || mask_heads == num_heads, "ncnnhip_attention_f32: the mask is shared (1) or one per head");
    if (attention_fewq_applies(head_dim, src_seqlen, dst_seqlen) && workspace_dev
        && workspace_bytes >= attention_fewq_workspace_bytes(num_heads, head_dim, src_seqlen, dst_seqlen))
    {
        const int v_vec_ok = (kv_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(vt_dev) & 15) == 0) ? 1 : 0;
        const int splits = (dst_seqlen + FEWQ_KEYS - 1) / FEWQ_KEYS; // (src_seqlen <= ATT_TQ: one group of queries)
        hipStream_t st = as_stream(stream);
        const dim3 grid((unsigned)splits, (unsigned)num_heads);
        const int mh = mask_dev ? mask_heads : 0;
#define LAUNCH_FEWQ(HD_, TQ_)                                                                                                                                      \
    hipLaunchKernelGGL((attention_fewq_split_hd_kernel<HD_, TQ_>), dim3(grid.x * grid.y), dim3(256), 0, st, q_dev, q_stride, q_scale, kt_dev, vt_dev, kv_stride, mask_dev, mh, src_seqlen, \
                       dst_seqlen, v_vec_ok, (float*)workspace_dev, append_k, append_v, append_stride, past, splits)
#define LAUNCH_FEWQ_HD(HD_)         \
    do                              \
    {                               \
        if (src_seqlen == 1)        \
            LAUNCH_FEWQ(HD_, 1);    \
        else if (src_seqlen == 2)   \
            LAUNCH_FEWQ(HD_, 2);    \
        else                        \
            LAUNCH_FEWQ(HD_, 4);    \
    } while (0)
        const bool one_row = (long long)splits * num_heads <= 1 << 23; // of workgroups
        if (head_dim == 32 && one_row)
            LAUNCH_FEWQ_HD(32);
        else if (head_dim == 64 && one_row)
            LAUNCH_FEWQ_HD(64);
        else if (head_dim == 96 && one_row)
            LAUNCH_FEWQ_HD(96);
        else if (head_dim == 128 && one_row)
            LAUNCH_FEWQ_HD(128);
        else
            hipLaunchKernelGGL(attention_fewq_split_kernel, grid, dim3(256), 0, st, q_dev, q_stride, q_scale, kt_dev, vt_dev, kv_stride, mask_dev, mh, head_dim, src_seqlen,
                               dst_seqlen, v_vec_ok, (float*)workspace_dev, append_k, append_v, append_stride, past);
#undef LAUNCH_FEWQ_HD
#undef LAUNCH_FEWQ
        hipLaunchKernelGGL(attention_fewq_merge_kernel, dim3((unsigned)num_heads, 1, (unsigned)((src_seqlen * head_dim + 63) / 64)), dim3(256), 0, st,
                           (const float*)workspace_dev, splits, head_dim, num_heads * head_dim, src_seqlen, out_dev);
        return launch_status("attention_fewq_split_kernel");
    }
    hipStream_t st = as_stream(stream);
    const int e = num_heads * head_dim, mh = mask_dev ? mask_heads : 0, query_blocks = (src_seqlen + 31) / 32;
    // 16-byte loads of the values need the rows and the start aligned
    const int v_vec_ok = (kv_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(vt_dev) & 15) == 0) ? 1 : 0;
    const unsigned units = (unsigned)query_blocks * (unsigned)num_heads;
    // enough workgroups for the merge: the outputs of a unit shared out over up to 8 of them
    const auto merge = [&](const float* partial, int splits) {
        unsigned shares = 1;
        while (shares < 8 && units * shares < 256 && (unsigned)(32 * head_dim) / (shares * 2) >= 256) shares *= 2;
        hipLaunchKernelGGL(attention_merge_kernel, dim3(units, shares), dim3(256), 0, st, partial, query_blocks, splits, head_dim, e, src_seqlen,
                           out_dev);
    };
    if (attention_bf16x3_applies(num_heads, head_dim, src_seqlen, dst_seqlen) && workspace_dev && (reinterpret_cast<uintptr_t>(workspace_dev) & 15) == 0
        && workspace_bytes >= attention_bf16x3_bytes(num_heads, head_dim, src_seqlen, dst_seqlen))
    {
        int keys_per_split;
        const int splits = attention_bf16x3_splits(num_heads, head_dim, src_seqlen, dst_seqlen, keys_per_split);
        uint4* frags = static_cast<uint4*>(workspace_dev);
        float* partial = reinterpret_cast<float*>(static_cast<char*>(workspace_dev) + attention_frags_bytes(num_heads, head_dim, dst_seqlen));
        const dim3 tiles((unsigned)((dst_seqlen + 31) / 32), (unsigned)num_heads), grid(units * (unsigned)splits);
#define LAUNCH_ATT(HD_)                                                                                                                                            \
    do                                                                                                                                                             \
    {                                                                                                                                                              \
        hipLaunchKernelGGL(attention_split_kernel<HD_>, tiles, dim3(256), 0, st, kt_dev, vt_dev, kv_stride, dst_seqlen, append_k, append_v, append_stride, past, frags); \
        hipLaunchKernelGGL(attention_bf16x3_kernel<HD_>, grid, dim3(256), 0, st, q_dev, kt_dev, vt_dev, frags, mask_dev, mh, e, src_seqlen, dst_seqlen, kv_stride,  \
                           out_dev, v_vec_ok, keys_per_split, partial, q_stride, q_scale, query_blocks, splits);                                 \
    } while (0)
        if (head_dim == 32)
            LAUNCH_ATT(32);
        else if (head_dim == 64)
            LAUNCH_ATT(64);
        else if (head_dim == 96)
            LAUNCH_ATT(96);
        else
            LAUNCH_ATT(128);
#undef LAUNCH_ATT
        if (splits > 1) merge(partial, splits);
        return launch_status("attention_bf16x3_kernel");
    }
    if (append_k)
    {
        // the other kernels read a finished cache: the new columns are written by a launch of their own
        const int rc = ncnnhip_transpose_pair_f32(append_k, append_v, append_stride, dst_seqlen - past, e, kt_dev + past, vt_dev + past, kv_stride, stream);
        if (rc != NCNNHIP_OK) return rc;
    }
    if (head_dim % 32 == 0 && head_dim <= 128)
    {
        // few queries (decoding): split the keys over workgroups when the caller brought the scratch for it
        int splits = attention_key_splits(num_heads, src_seqlen, dst_seqlen);
        if (splits > 1 && (!workspace_dev || workspace_bytes < attention_records_bytes(num_heads, head_dim, src_seqlen, dst_seqlen))) splits = 1;
        int keys_per_split = 0;
        if (splits > 1)
        {
            keys_per_split = ((dst_seqlen + splits - 1) / splits + 31) / 32 * 32;
            splits = (dst_seqlen + keys_per_split - 1) / keys_per_split;
        }
        dim3 grid((unsigned)query_blocks, (unsigned)num_heads, (unsigned)(splits > 1 ? splits : 1));
        if (splits <= 1) keys_per_split = 0;
        float* partial = (float*)workspace_dev;
#define LAUNCH_ATT(HD_)                                                                                                                                  \
    hipLaunchKernelGGL(attention_f32_mfma_kernel<HD_>, grid, dim3(256), 0, st, q_dev, kt_dev, vt_dev, mask_dev, mh, e, src_seqlen, dst_seqlen, kv_stride, \
                       out_dev, v_vec_ok, keys_per_split, partial, q_stride, q_scale)
        if (head_dim == 32)
            LAUNCH_ATT(32);
        else if (head_dim == 64)
            LAUNCH_ATT(64);
        else if (head_dim == 96)
            LAUNCH_ATT(96);
        else
            LAUNCH_ATT(128);
#undef LAUNCH_ATT
        if (keys_per_split > 0) merge(partial, splits);
        return launch_status("attention_f32_mfma_kernel");
    }
    const size_t lds = (size_t)ATT_TQ * ((size_t)head_dim + (size_t)dst_seqlen) * sizeof(float);
    NCNNHIP_REQUIRE(lds <= 65536, "ncnnhip_attention_f32: head_dim %d is not 32/64/96/128 and head_dim + dst_seqlen = %d exceeds the 4096 the general kernel keeps in LDS",
                    head_dim, head_dim + dst_seqlen);
    dim3 grid((unsigned)((src_seqlen + ATT_TQ - 1) / ATT_TQ), (unsigned)num_heads);
    hipLaunchKernelGGL(attention_f32_kernel, grid, dim3(256), lds, as_stream(stream), q_dev, kt_dev, vt_dev, mask_dev, mask_dev ? mask_heads : 0, head_dim,
                       num_heads * head_dim, src_seqlen, dst_seqlen, kv_stride, out_dev, q_stride, q_scale);
    return launch_status("attention_f32_kernel");
}
