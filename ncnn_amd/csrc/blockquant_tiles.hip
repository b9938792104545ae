// Block-quantised Gemm on many rows of fp32 activations (prefill, attention projections), weights in blocks of 64 or 128: the activations
// are split into two fp16 numbers by a pass of its own, then a workgroup multiplies 64 of their rows with 128 weight rows on
// v_mfma_f32_32x32x16_f16.
//
// Two fp16 numbers hold 23 bits of an activation, one less than fp32, and make two products of what were three with the exact split into bf16; with a third fewer
// roundings in the sums the error against 64 bits is smaller than it was: N(0, 1) rows, K 1024 1.05e-7 for 1.09e-7, 4096 1.22 for 1.26, 11008 1.54 for 1.57, 12800 in
// blocks of 128 1.61 for 1.64; one column in 97 300 times the others 1.40 for 1.39.  (The low parts of a step first: 1.20 at K = 4096, 1.59 at 11008.)
//
// A wavefront multiplies 64 activation rows with 64 weight rows and a workgroup holds four groups of two, each with a quarter of K: a weight
// is converted to fp16 once for 64 rows (with 32, as blockquant.hip's kernels have it, the vector unit is as busy as the matrix cores), and
// 256 tiles of 64 x 128, a prefill of 512 rows of 4096, still put two wavefronts on every SIMD.
// Bound by the matrix cores' issue at the 1.79 GHz they sustain on all units, and by the fills: half a K step is 571 ns of products for the two wavefronts of a SIMD and takes
// 921; without the fills (48 KB a unit, 13 TB/s on all of them) 700, without the vector instructions 770.  Around the 30 us of steps that 64 x 128 results of K = 4096 take
// stand 0.5 of first loads, 1.3 of the groups' exchange and 1.5 of results.  us with the split pass, 8 bits in blocks of 64, three bf16 numbers -> here: 512 x 4096 x 4096
// 60.7 -> 46.6, 512 x 4096 x 11008 133 -> 101, 512 x 11008 x 4096 145 -> 114, 1500 x 3072 x 1024 52.9 -> 43.9, 1500 x 1024 x 1024 24.1 -> 21.8; 1024 x 4096 x 4096 at 6
// bits 111 -> 86.  (One barrier a stage and operands read a stage ahead, between the products, instead of two wavefronts that read and multiply in turn: 49.8, as the
// fills are what it waits for.  Weights and loads all before the products, activations requested half a stage later, two groups and two workgroups to a
// unit: all slower with three products.)
#include <atomic>

#include "blockquant.h"

#define AS1 __attribute__((address_space(1)))
#define AS3 __attribute__((address_space(3)))
#define WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(0x0F70 | ((n) & 15) | ((((n) >> 4) & 3) << 14))

namespace ncnnhip {

typedef float v16f_bq __attribute__((ext_vector_type(16)));

// ---- the activations in operand order ----
// A row, times the power of two that takes its largest finite value into [2^14, 2^15), becomes hi + lo in fp16: 23 bits of a value of 24, and of values below 2^-17 of
// the row's largest what lies above 2^-40 of it.  The row's factor back goes to `back`; infinities and NaNs travel in hi alone.
// A stage is half a K step: of the 16-byte pieces the packed weights keep for four K groups (two chunks of 8 each) those of groups 2 h and
// 2 h + 1.  [row block of 64][K step][h] [32-row group][chunk c of the piece][part] 64 lanes x 16 bytes: lane = row l % 32, K group 2 h + l / 32.
// Rows beyond M and K beyond the last are zeros.  One workgroup: SPLIT_ROWS whole rows, so that their factors are known, and as many workgroups as that gives: 512 rows
// are 256 of them, one to a unit (bound by memory latency: each wavefront has its loads in flight once).  What it writes are 32-byte pieces; the four workgroups of a
// 128-byte line run on one die, so that its L2 puts the line together.
// A wavefront, of 16 or as many as there are spans of 256 columns, takes the spans in turn and keeps the first KEEP of its own in registers between the two passes.
// us, a decoder layer of 4096 / 11008, seven Gemms and as many of these, workgroups of four rows / here: 150 rows 367 / 354, 512 514.6 / 510.3; of 1024 / 2816, 1500 rows
// 213.1 / 209.9; of 2048 / 5504, 700 rows 257.8 / 256.5 (258.6 with four spans kept where there are no more than two).
constexpr int SPLIT_ROWS = 2, SPLIT_LINE = 8 / SPLIT_ROWS, SPLIT_SPAN = 512 / SPLIT_ROWS, SPLIT_WAVES = 16; // LINE: workgroups that write the same 128-byte lines
template<bool HALVES, int KEEP>
__global__ __launch_bounds__(64 * SPLIT_WAVES) void blockquant_split_tiles_kernel(const float* __restrict__ a, size_t a_stride, int M, int K, int kblocks,
                                                                                  const float* __restrict__ in_scales, uint4* __restrict__ frags, float* __restrict__ back)
{
    __shared__ unsigned tops[SPLIT_WAVES][SPLIT_ROWS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane % SPLIT_ROWS;
    const int turn = (int)blockIdx.x % (8 * SPLIT_LINE), share = (int)blockIdx.x - turn + (turn & 7) * SPLIT_LINE + (turn >> 3); // (the grid is whole turns)
    const int row = share * SPLIT_ROWS + r, waves = blockDim.x >> 6;
    const auto load = [&](int span, float (&x)[8]) {
        const int k = span * SPLIT_SPAN + lane / SPLIT_ROWS * 8;
        const bool inside = row < M && k < K; // K % 16 == 0: a chunk of 8 is all in or all out
        const float* p = a + (inside ? (size_t)row * a_stride + k : (size_t)0);
#pragma unroll
        for (int j = 0; j < 8; j++) x[j] = p[j]; // a valid address either way (K >= 16)
        if (!inside)
        {
#pragma unroll
            for (int j = 0; j < 8; j++) x[j] = 0.f;
        }
        else if (in_scales)
        {
#pragma unroll
            for (int j = 0; j < 8; j++) x[j] = mul_rn(x[j], in_scales[k + j]);
        }
    };
    const int spans = (kblocks * 64 + SPLIT_SPAN - 1) / SPLIT_SPAN;
    unsigned top = 0; // the bits of the largest finite magnitude
    const auto look = [&](const float (&x)[8]) {
#pragma unroll
        for (int j = 0; j < 8; j++)
        {
            const unsigned b = __float_as_uint(x[j]) & 0x7FFFFFFFu;
            if (b < 0x7F800000u && b > top) top = b;
        }
    };
    float kept[KEEP][8];
#pragma unroll
    for (int u = 0; u < KEEP; u++) load(wave + u * waves, kept[u]);
#pragma unroll
    for (int u = 0; u < KEEP; u++) look(kept[u]);
    for (int span = wave + KEEP * waves; span < spans; span += waves)
    {
        float x[8];
        load(span, x);
        look(x);
    }
#pragma unroll
    for (int d = SPLIT_ROWS; d < 64; d *= 2)
    {
        const unsigned o = (unsigned)__shfl_xor((int)top, d);
        if (o > top) top = o;
    }
    if (lane < SPLIT_ROWS) tops[wave][lane] = top;
    __syncthreads();
    for (int w = 0; w < waves; w++)
        if (tops[w][r] > top) top = tops[w][r];
    int shift = top ? 14 + 127 - (int)(top >> 23) : 0;
    if (shift > 126) shift = 126; // both factors are normal numbers
    const float factor = __uint_as_float((unsigned)(127 + shift) << 23);
    if (wave == 0 && lane < SPLIT_ROWS) back[row] = __uint_as_float((unsigned)(127 - shift) << 23);

    const auto store = [&](int span, const float (&x)[8]) {
        const int chunk_of_row = span * (SPLIT_SPAN / 8) + lane / SPLIT_ROWS, kb = chunk_of_row >> 3, chunk = chunk_of_row & 7;
        if (kb >= kblocks) return;
        // chunk = HALVES ? 2 h + hh + 4 c : 2 (2 h + hh) + c
        const int c = HALVES ? chunk >> 2 : chunk & 1, hh = HALVES ? chunk & 1 : (chunk >> 1) & 1, h = HALVES ? (chunk >> 1) & 1 : chunk >> 2;
        union
        {
            v8h h8;
            uint4 u;
        } hi, lo;
#pragma unroll
        for (int j = 0; j < 8; j++)
        {
            const float v = x[j] * factor;
            hi.h8[j] = (_Float16)v;
            const bool finite = (__float_as_uint(v) & 0x7F800000u) != 0x7F800000u;
            lo.h8[j] = (_Float16)(finite ? v - (float)hi.h8[j] : 0.f);
        }
        uint4* to = frags + ((((size_t)(row >> 6) * kblocks + kb) * 2 + h) * 8 + (((row >> 5) & 1) * 2 + c) * 2) * 64 + hh * 32 + (row & 31);
        to[0] = hi.u;
        to[64] = lo.u;
    };
#pragma unroll
    for (int u = 0; u < KEEP; u++) store(wave + u * waves, kept[u]);
    for (int span = wave + KEEP * waves; span < spans; span += waves)
    {
        float x[8];
        load(span, x);
        store(span, x);
    }
}

constexpr int TILES_STAGE = 8 * 1024; // bytes of activations
constexpr int tiles_weight_bytes(int bits) { return 8 * 64 * bits + 512; }
constexpr int KG = 4; // groups of two wavefronts
constexpr int tiles_lds_bytes(int bits) // the rings, or later the sums
{
    const int rings = KG * (2 * TILES_STAGE + 3 * tiles_weight_bytes(bits)), sums = (KG - 1) * KG * 2 * 4096;
    return rings > sums ? rings : sums;
}

// Each group has a ring of its own for two stages of activations (12 KB, read by both wavefronts) and three of weights and descales (read by
// the wavefront that fetched them, a stage ahead, and converted while it multiplies), filled straight from global memory as soon as
// the operands are in registers.  The last two groups run half a stage behind the first two, their neighbours on the same SIMDs: one
// reads while the other multiplies.
template<int BITS>
__global__ __launch_bounds__(KG * 128) void blockquant_tiles_kernel(const uint4* __restrict__ frags, const float* __restrict__ back, int M, int N, int kblocks, int ntiles,
                                                                   const unsigned char* __restrict__ wpk, const float4* __restrict__ dpk, const float* __restrict__ c,
                                                                   int bt, float alpha, float beta, float* __restrict__ out, size_t out_stride)
{
    constexpr int LOADS = 4 + (BITS == 4 ? 1 : BITS == 8 ? 2 : 3) + 1; // per wavefront and stage
    constexpr int HI_OFF = 2048, D_OFF = 8 * 64 * BITS, WSTAGE = tiles_weight_bytes(BITS), STEP_BYTES = 128 * BITS;
    constexpr int GROUP = 2 * TILES_STAGE + 3 * WSTAGE; // two slots of activations, three of weights
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds_tiles[];
    const int lane = threadIdx.x & 63, l32 = lane & 31, hh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), group = wave >> 1, ww = wave & 1;
    const int row0 = blockIdx.y * 64;
    const bool behind = group >= 2;

    // what this wavefront fetches: half of the fragments, and of the weights the four tiles of the 64 rows it multiplies (a tile beyond the
    // last reads the last one again and stores nothing); uniform base + 32-bit offset of the lane
    const int tile0 = (int)blockIdx.x * 8 + ww * 4, tile_first = tile0 < ntiles ? tile0 : ntiles - 1;
    const auto tile_offset = [&](int t) { return (unsigned)((tile_first + t < ntiles ? tile_first + t : ntiles - 1) - tile_first) * (unsigned)kblocks; };
    const char* const abase = reinterpret_cast<const char*>(frags + ((size_t)blockIdx.y * kblocks * 16 + ww * 4) * 64);
    const char* const wbase = reinterpret_cast<const char*>(wpk) + (size_t)tile_first * kblocks * STEP_BYTES;
    const char* const dbase = reinterpret_cast<const char*>(dpk) + (size_t)tile_first * kblocks * 64;
    unsigned woff[3];
    if constexpr (BITS == 8)
    {
#pragma unroll
        for (int i = 0; i < 2; i++) woff[i] = tile_offset(2 * i + hh) * STEP_BYTES + l32 * 16;
    }
    else
    {
        woff[0] = tile_offset(lane >> 4) * STEP_BYTES + (lane & 15) * 16;
        if constexpr (BITS == 6) // the third dwords: 32 a tile and half
        {
#pragma unroll
            for (int i = 0; i < 2; i++) woff[1 + i] = tile_offset(2 * i + hh) * STEP_BYTES + 512 + l32 * 4;
        }
    }
    const unsigned doff = tile_offset(lane >> 4) * 64 + (lane & 15) * 4;
    const int iterations = (kblocks + KG - 1) / KG, first = group * iterations, last = kblocks - 1;
    unsigned char* const mine = lds_tiles + group * GROUP;
    // load i of a stage: 4 of activations (of half h of K step `at`; h is also their slot), the others of weights (of a later stage)
    const auto load_activations = [&](int at, int h, int i) {
        const char* from = abase + (size_t)((at < last ? at : last) * 2 + h) * TILES_STAGE;
        __builtin_amdgcn_global_load_lds((const AS1 void*)(from + (unsigned)(lane * 16 + i * 1024)), (AS3 void*)(mine + h * TILES_STAGE + (ww * 4 + i) * 1024), 16, 0, 0);
    };
    const auto load_weights = [&](int at, int h, int slot, int i) {
        const int kb = at < last ? at : last;
        unsigned char* st = mine + 2 * TILES_STAGE + slot * WSTAGE;
        const char* from = wbase + (size_t)kb * STEP_BYTES + h * (BITS == 8 ? 512 : 256);
        if (i == LOADS - 5)
            __builtin_amdgcn_global_load_lds((const AS1 void*)(dbase + (size_t)kb * 64 + doff), (AS3 void*)(st + D_OFF + ww * 256), 4, 0, 0);
        else if (BITS == 8)
            __builtin_amdgcn_global_load_lds((const AS1 void*)(from + woff[i]), (AS3 void*)(st + (ww * 2 + i) * 1024), 16, 0, 0);
        else if (i == 0)
            __builtin_amdgcn_global_load_lds((const AS1 void*)(from + woff[0]), (AS3 void*)(st + ww * 1024), 16, 0, 0);
        else
            __builtin_amdgcn_global_load_lds((const AS1 void*)(wbase + (size_t)kb * STEP_BYTES + h * 128 + woff[i]), (AS3 void*)(st + HI_OFF + ww * 512 + (i - 1) * 256), 4, 0, 0);
    };
    const auto issue_activations = [&](int at, int h) {
#pragma unroll
        for (int i = 0; i < 4; i++) load_activations(at, h, i);
    };
    const auto issue_weights = [&](int at, int h, int slot) {
#pragma unroll
        for (int i = 0; i < LOADS - 4; i++) load_weights(at, h, slot, i);
    };

    v16f_bq acc[4], t[4]; // 32 x 32 parts: activation rows q / 2, weight rows q % 2; lane = weight row, register r = activation row 8 (r / 4) + 4 hh + r % 4
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[q][r] = t[q][r] = 0.f;
    const unsigned lds_base = (unsigned)(uintptr_t)(AS3 unsigned char*)mine;
    const int wt = ww * 4 + (l32 >> 4), wl = hh * 16 + (l32 & 15); // the lane's weight row: tile and place of its piece, for the first 32 of the wavefront
    const unsigned a_at = lds_base + (unsigned)(lane * 16), w_at = lds_base + 2 * TILES_STAGE + (unsigned)(wt * (BITS == 8 ? 512 : 256) + wl * (BITS == 8 ? 16 : 8)),
                   hi_at = lds_base + 2 * TILES_STAGE + HI_OFF + (unsigned)(wt * 128 + wl * 4), d_at = lds_base + 2 * TILES_STAGE + D_OFF + (unsigned)(ww * 256 + l32 * 4);

    // LDS is read with hand-written instructions and waits: the compiler treats a direct-to-LDS load as a store to all of LDS and would
    // drain every load in flight in front of each read it emits itself.  A wait names the registers it covers as in/out operands.
    v4i_bq wq[2];
    v2i_bq wlo[2];
    int whi[2];
    float d[2] = {0.f, 0.f};
    const auto scale = [&]() {
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[q][r] = fmaf(t[q][r], d[q & 1], acc[q][r]);
    };
    const auto read_weights = [&](int slot) {
        const unsigned o = (unsigned)(slot * WSTAGE);
#pragma unroll
        for (int g = 0; g < 2; g++)
        {
            if constexpr (BITS == 8)
                asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(wq[g]) : "v"(w_at + o), "n"(g * 1024));
            else
                asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(wlo[g]) : "v"(w_at + o), "n"(g * 512));
            if constexpr (BITS == 6) asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(whi[g]) : "v"(hi_at + o), "n"(g * 256));
        }
    };
    const auto weights_here = [&]() {
#pragma unroll
        for (int g = 0; g < 2; g++)
        {
            if constexpr (BITS == 8)
                asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(wq[g]));
            else
                asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(wlo[g]));
            if constexpr (BITS == 6) asm volatile("" : "+v"(whi[g]));
        }
    };
    const auto convert = [&](v8h (&w)[2][2], int part) { // [32 weight rows][chunk], in four parts
        const int g = part >> 1, ch = part & 1;
        if constexpr (BITS == 8)
            w[g][ch] = bytes_to_halves(wq[g][2 * ch], wq[g][2 * ch + 1]);
        else if constexpr (BITS == 4)
            w[g][ch] = nibbles_to_halves((unsigned)wlo[g][ch]);
        else if (ch == 0)
            sixbit_to_halves((unsigned)wlo[g][0], (unsigned)wlo[g][1], (unsigned)whi[g], w[g][0], w[g][1]);
    };

    v8h w[2][2];
    issue_weights(first, 0, 0);
    issue_activations(first, 0);
    issue_weights(first, 1, 1);
    issue_activations(first, 1);
    issue_weights(first + 1, 0, 2);
    WAIT_VMCNT(2 * LOADS); // (each wavefront brings the weights that it multiplies itself)
    asm volatile("" ::: "memory");
    read_weights(0);
    weights_here();
#pragma unroll
    for (int i = 0; i < 4; i++) convert(w, i);
    int slot = 0; // of this stage's weights
    if (behind) __builtin_amdgcn_s_barrier();
    const auto stage = [&](int kb, auto half) {
        constexpr int h = decltype(half)::value;
        WAIT_VMCNT(LOADS);            // this wavefront's activations of the stage and weights of the next have landed, a stage of loads may still be on its way
        __builtin_amdgcn_s_barrier(); // and everybody else's
        asm volatile("" ::: "memory");
        const int next = slot == 2 ? 0 : slot + 1;
        union Act
        {
            v4i_bq i4;
            v8h b;
        };
        Act y[8];
#pragma unroll
        for (int i = 0; i < 8; i++) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(y[i].i4) : "v"(a_at), "n"(h * TILES_STAGE + i * 1024));
        read_weights(next);
        if constexpr (h == 0)
        {
            __builtin_amdgcn_sched_barrier(0);
            scale(); // the step before, while the operands come
            __builtin_amdgcn_sched_barrier(0);
            const unsigned o = (unsigned)(slot * WSTAGE);
#pragma unroll
            for (int g = 0; g < 2; g++) asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(d[g]) : "v"(d_at + o), "n"(g * 128));
        }
#pragma unroll
        for (int i = 0; i < 8; i++) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(y[i].i4));
        weights_here();
        if constexpr (h == 0) asm volatile("" : "+v"(d[0]), "+v"(d[1]));
        __builtin_amdgcn_s_barrier(); // both wavefronts of the group have read the stage
        asm volatile("" ::: "memory");
        if constexpr (h == 0)
        {
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int r = 0; r < 16; r++) t[q][r] = 0.f;
        }
        v8h wn[2][2]; // the next stage's
        // four rounds of four products; the loads and the conversions spread over them
#pragma unroll
        for (int c = 0; c < 4; c++)
        {
            const int ch = c / 2, p = c % 2;
#pragma unroll
            for (int i = c * LOADS / 4; i < (c + 1) * LOADS / 4; i++)
            {
                if (i < 4)
                    load_activations(kb + 1, h, i);
                else
                    load_weights(h == 0 ? kb + 1 : kb + 2, h ^ 1, slot, i - 4);
            }
#pragma unroll
            for (int q = 0; q < 4; q++) t[q] = __builtin_amdgcn_mfma_f32_32x32x16_f16(y[((q >> 1) * 2 + ch) * 2 + p].b, w[q & 1][ch], t[q], 0, 0, 0);
            convert(wn, c);
#pragma unroll
            for (int q = 0; q < 4; q++)
            {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (q < (c + 1) * LOADS / 4 - c * LOADS / 4) __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        slot = next;
#pragma unroll
        for (int g = 0; g < 2; g++)
#pragma unroll
            for (int ch = 0; ch < 2; ch++) w[g][ch] = wn[g][ch];
    };
    const int end = first + iterations < kblocks ? first + iterations : kblocks;
    for (int kb = first; kb < end; kb++)
    {
        stage(kb, std::integral_constant<int, 0>{});
        stage(kb, std::integral_constant<int, 1>{});
    }
    scale();
    for (int kb = end > first ? end : first; kb < first + iterations; kb++) // a group with fewer steps keeps the others company
    {
#pragma unroll
        for (int i = 0; i < 4; i++) __builtin_amdgcn_s_barrier();
    }
    if (!behind) __builtin_amdgcn_s_barrier(); // the others' last half stage
    WAIT_VMCNT(0);                                       // the surplus loads of the last stages must not outlive the workgroup's LDS

    // the groups hand their sums over through LDS: part q is finished by group q, the others leave theirs in [part][group][wavefront][register / 4][lane]
    typedef float v4f_t __attribute__((ext_vector_type(4)));
    v4f_t* meet = reinterpret_cast<v4f_t*>(lds_tiles);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; q++)
        if (q != group)
        {
            v4f_t* to = meet + ((q * (KG - 1) + (group < q ? group : group - 1)) * 2 + ww) * 256 + lane;
#pragma unroll
            for (int e = 0; e < 4; e++) to[e * 64] = v4f_t{acc[q][4 * e], acc[q][4 * e + 1], acc[q][4 * e + 2], acc[q][4 * e + 3]};
        }
    // what the part's results need from memory is on its way while the groups meet (read behind their sums it was 1.5 us of a workgroup's time)
    const int j = (tile0 + 2 * (group & 1)) * 16 + l32, i0 = row0 + (group >> 1) * 32 + 4 * hh; // result r: row i0 + 8 (r / 4) + r % 4 (`back` is padded to 64 rows)
    v4f_t factor[4];
#pragma unroll
    for (int e = 0; e < 4; e++) factor[e] = *reinterpret_cast<const v4f_t*>(back + i0 + 8 * e);
    const bool of_column = bt == 0 || bt == 4;
    const float addend = of_column && j < N ? mul_rn(load_c(c, bt, 0, j, N), beta) : 0.f;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; q++)
    {
        if (q != group) continue;
#pragma unroll
        for (int s = 0; s < KG - 1; s++)
        {
            const v4f_t* from = meet + ((q * (KG - 1) + s) * 2 + ww) * 256 + lane;
#pragma unroll
            for (int e = 0; e < 4; e++)
            {
                const v4f_t v = from[e * 64];
#pragma unroll
                for (int o = 0; o < 4; o++) acc[q][4 * e + o] += v[o];
            }
        }
        if (j >= N) continue;
#pragma unroll
        for (int r = 0; r < 16; r++)
        {
            const int i = i0 + 8 * (r >> 2) + (r & 3);
            if (i < M)
            {
                float v = acc[q][r] * factor[r >> 2][r & 3];
                if (of_column)
                    v = add_rn(addend, v);
                else if (bt >= 0)
                    v = add_rn(mul_rn(load_c(c, bt, i, j, N), beta), v);
                out[(size_t)i * out_stride + j] = mul_rn(v, alpha);
            }
        }
    }
}

int launch_blockquant_tiles(const float* a, size_t a_stride, int M, int N, int K, int bits, const unsigned char* wpk, const float4* dpk, const float* in_scales,
                            const float* c, int bt, float alpha, float beta, float* out, size_t out_stride, void* workspace, hipStream_t st)
{
    const int kblocks = (K + 63) / 64, ntiles = (N + 15) / 16, blocks = (M + 63) / 64;
    uint4* frags = static_cast<uint4*>(workspace);
    float* back = reinterpret_cast<float*>(frags + (size_t)blocks * kblocks * 1024); // 4 bytes a value, and the rows' factors behind them
    const dim3 grid((unsigned)((ntiles + 7) / 8), (unsigned)blocks);
    const int spans = (kblocks * 64 + SPLIT_SPAN - 1) / SPLIT_SPAN, waves = spans < SPLIT_WAVES ? spans : SPLIT_WAVES;
#define SPLIT(HALVES_, KEEP_) \
    hipLaunchKernelGGL((blockquant_split_tiles_kernel<HALVES_, KEEP_>), dim3((unsigned)(blocks * (64 / SPLIT_ROWS))), dim3((unsigned)(64 * waves)), 0, st, a, a_stride, M, K, kblocks, in_scales, frags, back)
    const int keep = (spans + SPLIT_WAVES - 1) / SPLIT_WAVES; // what a wavefront keeps, up to three (K = 12288)
    if (keep == 1 && bits == 8)
        SPLIT(false, 1);
    else if (keep == 1)
        SPLIT(true, 1);
    else if (keep == 2 && bits == 8)
        SPLIT(false, 2);
    else if (keep == 2)
        SPLIT(true, 2);
    else if (bits == 8)
        SPLIT(false, 3);
    else
        SPLIT(true, 3);
#undef SPLIT
#define TILES(BITS_)                                                                                                                                          \
    do                                                                                                                                                             \
    {                                                                                                                                                              \
        auto kernel = blockquant_tiles_kernel<BITS_>;                                                                                                         \
        static std::atomic<unsigned char> raised[64];                                                                                                              \
        int device = 0;                                                                                                                                            \
        NCNNHIP_CHECK(hipGetDevice(&device));                                                                                                                      \
        if (device < 0 || device >= 64 || !raised[device].load(std::memory_order_acquire))                                                                         \
        {                                                                                                                                                          \
            NCNNHIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));                     \
            if (device >= 0 && device < 64) raised[device].store(1, std::memory_order_release);                                                                    \
        }                                                                                                                                                          \
        hipLaunchKernelGGL(kernel, grid, dim3(KG * 128), tiles_lds_bytes(BITS_), st, frags, back, M, N, kblocks, ntiles, wpk, dpk, c, bt, alpha, beta, out,      \
                           out_stride);                                                                                                                            \
    } while (0)
    if (bits == 8)
        TILES(8);
    else if (bits == 6)
        TILES(6);
    else
        TILES(4);
#undef TILES
    return launch_status("blockquant_tiles_kernel");
}

} // namespace ncnnhip
