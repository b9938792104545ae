// Block-quantised Gemm on many activation rows, fp16 (from 5, by weights: many_rows_f16) or fp32 (many_rows_f32): every weight is read
// once for up to 64 (fp32: 32) rows.
//
// The few-row kernels (blockquant.hip) multiply 16 rows per pass over the weights; 48 rows were three passes of a launch each.
// Here a workgroup owns RT tiles of 16 weight rows and MG groups of 16 activation rows and deals the K steps of 64 out to its
// wavefronts, each a run of its own.  A wavefront streams what a step needs -- MG x 16 rows of 128 or 256 bytes, its RT tiles
// and their descales -- from global memory straight into LDS, into a ring of two stages that belongs to it alone: no barrier and
// no other wavefront stands in its way, and the eight of a workgroup keep about 80 KB in flight on a compute unit.  The sums
// of the wavefronts meet in LDS at the end.
//
// fp16: what bounds it is not the weights but the activations: every workgroup reads all M x K of them (393 KB for 48 rows of 4096)
// through its unit's L1, so MG and RT balance re-reading them against idle units (launch_blockquant_rows_f16).
// us per launch, 16 rows per pass -> here, weights from HBM, 4 bits in blocks of 64: 4096 x 4096 24 rows 11.9 -> 8.9, 48 rows 18.4 -> 10.8,
// 128 rows 45.9 -> 14.6; 11008 x 4096 48 rows 37.3 -> 16.8; 4096 x 11008 48 rows 102 -> 21.5; 8 bits 48 rows 4096 x 4096 20.0 -> 11.3,
// 11008 x 4096 42.6 -> 19.1, 4096 x 11008 48.0 -> 23.4.
// fp32: an activation becomes three bf16 numbers that add up to it exactly (split_bf16x3) when it has been read from LDS, and a
// step's product six matrix-core instructions instead of two.  Bound by vector issue: the split (88 instructions per 16 rows and step), the
// weights' conversion (30 to 50 per tile and step), at about 5 cycles an instruction with two or three wavefronts per SIMD; neither a
// third stage nor activations that hit L1 every time made it quicker.  Against a pass that splits them beforehand and a kernel on the
// parts it saves that launch (5 us) and a third of the bytes.  us per call before (blockquant.hip's forms) -> here, 8 bits in blocks of 64:
// 4096 x 4096 16 rows 12.4 -> 10.7, 32 rows 20.1 -> 12.9, 64 rows 34 -> 17.5, 128 rows 41 -> 30; 11008 x 4096 16 rows 26.5 -> 16.6, 32
// rows 46 -> 26.5; 4096 x 11008 32 rows 45 -> 27, 128 rows 93 -> 66.
// Two wavefronts share a SIMD and the one that multiplies goes first (left to itself the SIMD serves its oldest, which ends up to 4 us
// before its neighbour and leaves it alone with its waits); the sums of a result are requested at once.  us a launch in a chain of them,
// before -> here: fp32 rows, 8 bits, 64 x 4096 x 4096 16.4 -> 15.7, 42 x 6880 x 5312 33.6 -> 32.3, 16 x 4096 x 4096 10.5 -> 10.1, 6 bits
// 100 x 1248 x 7296 24.6 -> 23.6; fp16 rows, the four launches of a decoder layer, 48 rows at 4 bits 54.2 -> 52.4; a K of 256 or 384 is 1 %
// slower, by the branch of its sums.  (Loads of the stage after the next as soon as a stage is in registers: 66.6 -> 68.6 for the layer.
// Without any loads its four launches take 48, without the products 50, with neither 29.)
// A lane must fetch along a row (eight lanes = one 128-byte line) and read in operand order (lane = row), so the chunks of a row
// are swizzled on the source side: chunk c of row r lands at position c ^ ((r / 2) % 8), conflict-free both ways.
#include <atomic>

#include "blockquant.h"

#define AS1 __attribute__((address_space(1)))
#define AS3 __attribute__((address_space(3)))

namespace ncnnhip {

// s_waitcnt immediate that waits for vmcnt <= n only (gfx9 encoding)
#define WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(0x0F70 | ((n) & 15) | ((((n) >> 4) & 3) << 14))

constexpr int rows_stage_bytes(int bits, int mg, int rt, int split, int ain)
{
    return mg * 1024 * ain + rt * 128 * bits + rt * (64 << split) + (ain == 4 ? 256 : 0);
}

// LDS a wavefront needs: its ring, later its sums
constexpr int rows_wave_bytes(int bits, int mg, int rt, int split, int ain)
{
    return 2 * rows_stage_bytes(bits, mg, rt, split, ain) > rt * mg * 1024 ? 2 * rows_stage_bytes(bits, mg, rt, split, ain) : rt * mg * 1024;
}
// Wavefronts of a workgroup, of which a compute unit holds one.  (Always 8 for one group of fp32 rows: the order of its sums is then the
// same whatever RT a launch takes, so that several matrices in one call get the bits of single calls.  Twelve, where they fit, took 4096 x
// 4096 16 rows from 10.9 to 10.7 us.)
constexpr int rows_waves(int bits, int mg, int rt, int split, int ain)
{
    const int fit = 160 * 1024 / rows_wave_bytes(bits, mg, rt, split, ain);
    return fit >= 8 ? 8 : fit;
}

template<int BITS>
__device__ __forceinline__ void fields_to_halves(const v4i_bq& wq, const v2i_bq& wlo, int whi, v8h& wa, v8h& wb)
{
    if (BITS == 8)
    {
        wa = bytes_to_halves(wq[0], wq[1]);
        wb = bytes_to_halves(wq[2], wq[3]);
    }
    else if (BITS == 4)
    {
        wa = nibbles_to_halves((unsigned)wlo[0]);
        wb = nibbles_to_halves((unsigned)wlo[1]);
    }
    else
        sixbit_to_halves((unsigned)wlo[0], (unsigned)wlo[1], (unsigned)whi, wa, wb);
}
template<int BITS>
__device__ __forceinline__ void fields_to_bf16(const v4i_bq& wq, const v2i_bq& wlo, int whi, v8bf& wa, v8bf& wb)
{
    if (BITS == 8)
    {
        wa = bytes_to_bf16((unsigned)wq[0], (unsigned)wq[1]);
        wb = bytes_to_bf16((unsigned)wq[2], (unsigned)wq[3]);
    }
    else if (BITS == 4)
    {
        wa = nibbles_to_bf16((unsigned)wlo[0]);
        wb = nibbles_to_bf16((unsigned)wlo[1]);
    }
    else
        sixbit_to_bf16((unsigned)wlo[0], (unsigned)wlo[1], (unsigned)whi, wa, wb);
}

// 8 floats -> three bf16 parts each that add up to it exactly (split_bf16x3).  FAST leaves out the check of every value: an infinity
// makes NaNs of its lesser parts; the caller then sees a NaN in its sums and repeats them with the check.
template<bool FAST>
__device__ __forceinline__ void split8_bf16x3(const float* x, v8bf (&out)[3])
{
    union
    {
        unsigned i[4];
        v8bf h;
    } p[3];
#pragma unroll
    for (int e = 0; e < 4; e++)
    {
        unsigned h[2][3];
#pragma unroll
        for (int o = 0; o < 2; o++)
        {
            const float v = x[2 * e + o];
            if (FAST)
            {
                h[o][0] = __float_as_uint(v);
                const float r1 = v - __uint_as_float(h[o][0] & 0xFFFF0000u);
                h[o][1] = __float_as_uint(r1);
                h[o][2] = __float_as_uint(r1 - __uint_as_float(h[o][1] & 0xFFFF0000u));
            }
            else
                split_bf16x3(v, h[o][0], h[o][1], h[o][2]);
        }
#pragma unroll
        for (int pn = 0; pn < 3; pn++) p[pn].i[e] = __builtin_amdgcn_perm(h[1][pn], h[0][pn], 0x07060302u);
    }
#pragma unroll
    for (int pn = 0; pn < 3; pn++) out[pn] = p[pn].h;
}

template<int BITS, bool HALVES, int SPLIT, int MG, int RT, int AIN>
__global__ __launch_bounds__(rows_waves(BITS, MG, RT, SPLIT, AIN) * 64) void blockquant_rows_kernel(const void* __restrict__ a_, size_t a_stride, int M_total, int K, int kblocks,
                                                                              int groups, int passes, const float* __restrict__ in_scales, BqMulti mm)
{
    static_assert(HALVES || (BITS == 8 && SPLIT == 0), "4- and 6-bit fields and blocks of 32 come in the halves layout");
    constexpr bool F32 = AIN == 4;
    constexpr int STEP_BYTES = 128 * BITS;   // one tile's weights for a step
    constexpr int DPER = 4 << SPLIT;         // its descales, in float4
    constexpr int G_BYTES = 1024 * AIN;      // a group of 16 activation rows: 128 or 256 bytes each
    constexpr int W_OFF = MG * G_BYTES, D_OFF = W_OFF + RT * STEP_BYTES, S_OFF = D_OFF + RT * DPER * 16;
    constexpr int STAGE = rows_stage_bytes(BITS, MG, RT, SPLIT, AIN);
    constexpr int ALOADS = MG * AIN; // of 1 KB: 8 rows of fp16, 4 of fp32
    constexpr int LOADS = ALOADS + RT + 1 + (F32 ? 1 : 0);
    constexpr int CHUNK = 16 / AIN; // activations in 16 bytes
    const unsigned char* a = static_cast<const unsigned char*>(a_);
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds_rows[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nwaves = blockDim.x >> 6;
    const int m = lane & 15, kg = lane >> 4;

    // the passes over one group of tiles follow each other on one die (workgroups are dealt to the 8 dies in turn)
    const int round = blockIdx.x / (8 * passes), in_round = blockIdx.x - round * 8 * passes;
    int group = round * 8 + (in_round & 7);
    const int row0 = (in_round >> 3) * MG * 16;
    if (group >= groups) return;
    int mat = 0; // tile_end counts groups of RT tiles here
    while (mat + 1 < mm.count && group >= mm.tile_end[mat]) mat++; // (all ends read at once: 1 to 2 % slower for one matrix, 0.3 % for two to four)
    group -= mat ? mm.tile_end[mat - 1] : 0;
    const int N = mm.N[mat], ntiles = (N + 15) >> 4;
    const int M = M_total - row0 < MG * 16 ? M_total - row0 : MG * 16;

    // this wavefront's K steps
    const int step0 = (int)((long long)kblocks * wave / nwaves), steps = (int)((long long)kblocks * (wave + 1) / nwaves) - step0;
    const int ragged = (K & 63) ? kblocks - 1 - step0 : -1; // the step K ends in (the last wavefront's; beyond the others' steps)

    // sources.  Activations: load i brings rows i * 8 .. + 8 of the pass, lane l row l / 8 and the chunk that belongs at position l % 8
    const int chunk0 = F32 ? (lane & 15) ^ (lane >> 4) : (lane & 7) ^ ((lane >> 4) & 7);
    auto chunk_k = [&](int i) { return (F32 ? chunk0 ^ ((i & 3) << 2) : chunk0 ^ ((i & 1) << 2)) * CHUNK; }; // where load i's chunk starts in the step
    const unsigned char* arow[ALOADS];
#pragma unroll
    for (int i = 0; i < ALOADS; i++)
    {
        const int r = F32 ? i * 4 + (lane >> 4) : i * 8 + (lane >> 3);
        arow[i] = a + ((size_t)(row0 + (r < M ? r : M - 1)) * a_stride + step0 * 64 + chunk_k(i)) * AIN;
    }
    // the input scales of the step (none: the first activations, which nobody reads there, so that the count of loads stays)
    const float* ssrc = F32 ? (in_scales ? in_scales + step0 * 64 + (lane & 15) * 4 : reinterpret_cast<const float*>(a)) : nullptr;
    const size_t s_step = F32 && in_scales ? 64 : 0;
    const unsigned char* wsrc[RT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
    {
        const int t = group * RT + rt;
        wsrc[rt] = mm.wpk[mat] + ((size_t)(t < ntiles ? t : ntiles - 1) * kblocks + step0) * STEP_BYTES + lane * 16;
    }
    // descales of the RT tiles side by side: lane l brings float4 l % DPER of tile l / DPER
    const int dtile = group * RT + lane / DPER;
    const float4* dsrc = mm.dpk[mat] + ((size_t)(dtile < ntiles ? dtile : ntiles - 1) * kblocks + step0) * DPER + lane % DPER;

    unsigned char* ring = lds_rows + wave * 2 * STAGE;
    auto issue = [&](int s, int slot) {
        unsigned char* st = ring + slot * STAGE;
        if (s != ragged)
        {
#pragma unroll
            for (int i = 0; i < ALOADS; i++)
                __builtin_amdgcn_global_load_lds((const AS1 void*)(arow[i] + (size_t)s * (64 * AIN)), (AS3 void*)(st + i * 1024), 16, 0, 0);
            if (F32 && lane < 16) __builtin_amdgcn_global_load_lds((const AS1 void*)(ssrc + s * s_step), (AS3 void*)(st + S_OFF), 16, 0, 0);
        }
        else
        {
            // K % 16 == 0: a chunk is all in or all out, and then replaced by the first of all
#pragma unroll
            for (int i = 0; i < ALOADS; i++)
                __builtin_amdgcn_global_load_lds((const AS1 void*)((step0 + s) * 64 + chunk_k(i) < K ? arow[i] + (size_t)s * (64 * AIN) : a), (AS3 void*)(st + i * 1024),
                                                 16, 0, 0);
            if (F32 && lane < 16)
                __builtin_amdgcn_global_load_lds((const AS1 void*)((step0 + s) * 64 + lane * 4 < K ? ssrc + s * s_step : reinterpret_cast<const float*>(a)),
                                                 (AS3 void*)(st + S_OFF), 16, 0, 0);
        }
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
            if (lane < STEP_BYTES / 16)
                __builtin_amdgcn_global_load_lds((const AS1 void*)(wsrc[rt] + (size_t)s * STEP_BYTES), (AS3 void*)(st + W_OFF + rt * STEP_BYTES), 16, 0, 0);
        if (lane < RT * DPER) __builtin_amdgcn_global_load_lds((const AS1 void*)(dsrc + (size_t)s * DPER), (AS3 void*)(st + D_OFF), 16, 0, 0);
    };

    v4f acc[RT][MG];
    const unsigned base = (unsigned)(uintptr_t)(AS3 unsigned char*)ring;
    // where the lane's 16 activations of a step lie: two chunks of fp16, four of fp32 (its place is XORed into the chunk number)
    constexpr int PARTS = F32 ? 4 : 2;
    unsigned rd_a[PARTS], rd_s[PARTS];
#pragma unroll
    for (int p = 0; p < PARTS; p++)
    {
        const int c = F32 ? (HALVES ? 2 * kg + (p & 1) + (p >> 1) * 8 : 4 * kg + p) : (HALVES ? kg + p * 4 : 2 * kg + p);
        rd_a[p] = base + m * (G_BYTES / 16) + ((c ^ (F32 ? m : (m >> 1) & 7)) << 4);
        rd_s[p] = base + S_OFF + (c << 4);
    }
    const unsigned rd_w = base + W_OFF + lane * (BITS == 8 ? 16 : 8), rd_w3 = base + W_OFF + 512 + lane * 4;
    const unsigned rd_d = base + D_OFF + kg * 16;
    // two descales a tile, four groups and six tiles: the descales of a tile are read while the one before is multiplied, or registers spill
    constexpr bool TILEWISE = F32 && MG == 2 && (RT == 4 || (RT == 3 && SPLIT)); // (fp32 rows: both groups split, then tile by tile; three tiles with one descale fit)
    constexpr bool LATE = SPLIT && ((!F32 && MG == 4 && RT == 6) || TILEWISE);
    auto read_descales = [&](int rt, unsigned at, v4i_bq (&dq0)[RT], v4i_bq (&dq1)[RT]) {
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dq0[rt]) : "v"(rd_d + at), "n"(rt * DPER * 16));
        if (SPLIT) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dq1[rt]) : "v"(rd_d + at), "n"(rt * DPER * 16 + 64));
    };

    for (bool careful = false;; careful = true)
    {
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
#pragma unroll
            for (int g = 0; g < MG; g++) acc[rt][g] = v4f{0.f, 0.f, 0.f, 0.f};
        issue(0, 0);
        for (int s = 0; s < steps; s++)
        {
            __builtin_amdgcn_s_setprio(0); // the neighbour on the SIMD multiplies first
            const unsigned at = (unsigned)((s & 1) * STAGE);
            // the stage multiplied in the turn before has been read (its reads were waited for): the next loads go there
            issue(s + 1 < steps ? s + 1 : s, (s + 1) & 1);
            WAIT_VMCNT(LOADS);
            asm volatile("" ::: "memory");
            if (s == ragged)
            {
                // zeros in place of the chunks beyond K (and of their input scales): their weights are zero, but zero times an infinity is not
                const v4i_bq zeros = {0, 0, 0, 0};
#pragma unroll
                for (int i = 0; i < ALOADS; i++)
                    if ((step0 + s) * 64 + chunk_k(i) >= K) asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(base + at + lane * 16), "v"(zeros), "n"(i * 1024) : "memory");
                if (F32 && lane < 16 && (step0 + s) * 64 + lane * 4 >= K) asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(base + at + lane * 16), "v"(zeros), "n"(S_OFF) : "memory");
            }
            // LDS is read with hand-written instructions and waits: the compiler takes a direct-to-LDS load for a store to all of LDS
            // and would wait for everything in flight in front of each read it emits itself.
            v4i_bq wq[RT], dq0[RT], dq1[RT];
            v2i_bq wlo[RT];
            int whi[RT];
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
            {
                if (BITS == 8)
                    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(wq[rt]) : "v"(rd_w + at), "n"(rt * STEP_BYTES));
                else
                    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(wlo[rt]) : "v"(rd_w + at), "n"(rt * STEP_BYTES));
                if (BITS == 6) asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(whi[rt]) : "v"(rd_w3 + at), "n"(rt * STEP_BYTES));
                if (!LATE || rt == 0) read_descales(rt, at, dq0, dq1);
            }
            union Act
            {
                v4i_bq i4;
                float f[4];
                v8h h;
            };
            Act x[MG][PARTS], sc[PARTS];
#pragma unroll
            for (int g = 0; g < MG; g++)
#pragma unroll
                for (int p = 0; p < PARTS; p++) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(x[g][p].i4) : "v"(rd_a[p] + at), "n"(g * G_BYTES));
            if (F32 && in_scales)
            {
#pragma unroll
                for (int p = 0; p < PARTS; p++) asm volatile("ds_read_b128 %0, %1" : "=v"(sc[p].i4) : "v"(rd_s[p] + at));
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (F32)
            {
#pragma unroll
                for (int p = 0; p < PARTS; p++) asm volatile("" : "+v"(sc[p].i4));
            }
#pragma unroll
            for (int g = 0; g < MG; g++)
#pragma unroll
                for (int p = 0; p < PARTS; p++) asm volatile("" : "+v"(x[g][p].i4));
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
            {
                if (BITS == 8)
                    asm volatile("" : "+v"(wq[rt]));
                else
                    asm volatile("" : "+v"(wlo[rt]));
                if (BITS == 6) asm volatile("" : "+v"(whi[rt]));
                if (LATE && rt > 0) continue;
                asm volatile("" : "+v"(dq0[rt]));
                if (SPLIT) asm volatile("" : "+v"(dq1[rt]));
            }
            __builtin_amdgcn_s_setprio(1);
            const v4f zero = {0.f, 0.f, 0.f, 0.f};
            if constexpr (!F32)
            {
                // tile by tile: with the tiles' operands and products side by side, as below, four groups and six tiles are 23 registers too
                // many, and a spilled one waits for every load in flight (twice the time)
#pragma unroll
                for (int rt = 0; rt < RT; rt++)
                {
                    v8h wa, wb;
                    if (LATE && rt + 1 < RT) read_descales(rt + 1, at, dq0, dq1);
                    fields_to_halves<BITS>(wq[rt], wlo[rt], whi[rt], wa, wb);
#pragma unroll
                    for (int g = 0; g < MG; g++)
                    {
                        v4f t0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(wa, x[g][0].h, zero, 0, 0, 0);
                        const v4f t1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(wb, x[g][1].h, SPLIT ? zero : t0, 0, 0, 0);
                        if (!SPLIT) t0 = t1;
#pragma unroll
                        for (int r = 0; r < 4; r++)
                        {
                            acc[rt][g][r] = fmaf(t0[r], __int_as_float(dq0[rt][r]), acc[rt][g][r]);
                            if (SPLIT) acc[rt][g][r] = fmaf(t1[r], __int_as_float(dq1[rt][r]), acc[rt][g][r]);
                        }
                    }
                    if (LATE && rt + 1 < RT)
                    {
                        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(dq0[rt + 1]), "+v"(dq1[rt + 1]));
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
            else
            {
                auto split_group = [&](int g, v8bf (&ya)[3], v8bf (&yb)[3]) {
                    float v[16];
#pragma unroll
                    for (int p = 0; p < PARTS; p++)
#pragma unroll
                        for (int e = 0; e < 4; e++) v[p * 4 + e] = x[g][p].f[e];
                    if (in_scales)
                    {
#pragma unroll
                        for (int p = 0; p < PARTS; p++)
#pragma unroll
                            for (int e = 0; e < 4; e++) v[p * 4 + e] = mul_rn(v[p * 4 + e], sc[p].f[e]);
                    }
                    if (careful)
                    {
                        split8_bf16x3<false>(v, ya);
                        split8_bf16x3<false>(v + 8, yb);
                    }
                    else
                    {
                        split8_bf16x3<true>(v, ya);
                        split8_bf16x3<true>(v + 8, yb);
                    }
                };
                // One chain for the whole step: the least parts first, so that only two of its six roundings are at the sum's own size
                // (relative error of 4096 x 4096 against 64 bits 9.2e-8 -> 7.1e-8); a chain of three is better begun with the
                // greatest (blocks of 32, 4 bits: 8.7e-8 against 9.1e-8).
                auto product = [&](v4f& t0, v4f& t1, const v8bf& wa, const v8bf& wb, const v8bf (&ya)[3], const v8bf (&yb)[3], int i) {
                    const int pn = SPLIT ? i : 2 - i;
                    t0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa, ya[pn], i ? t0 : zero, 0, 0, 0);
                    if (SPLIT)
                        t1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb, yb[pn], i ? t1 : zero, 0, 0, 0);
                    else
                        t0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb, yb[pn], t0, 0, 0, 0);
                };
                auto add = [&](int rt, int g, const v4f& t0, const v4f& t1) {
#pragma unroll
                    for (int r = 0; r < 4; r++)
                    {
                        acc[rt][g][r] = fmaf(t0[r], __int_as_float(dq0[rt][r]), acc[rt][g][r]);
                        if (SPLIT) acc[rt][g][r] = fmaf(t1[r], __int_as_float(dq1[rt][r]), acc[rt][g][r]);
                    }
                };
                if constexpr (TILEWISE)
                {
                    v8bf ya[MG][3], yb[MG][3];
#pragma unroll
                    for (int g = 0; g < MG; g++) split_group(g, ya[g], yb[g]);
#pragma unroll
                    for (int rt = 0; rt < RT; rt++)
                    {
                        v8bf wa, wb;
                        v4f t0[MG], t1[MG];
                        if (LATE && rt + 1 < RT) read_descales(rt + 1, at, dq0, dq1);
                        fields_to_bf16<BITS>(wq[rt], wlo[rt], whi[rt], wa, wb);
#pragma unroll
                        for (int i = 0; i < 3; i++)
#pragma unroll
                            for (int g = 0; g < MG; g++) product(t0[g], t1[g], wa, wb, ya[g], yb[g], i);
#pragma unroll
                        for (int g = 0; g < MG; g++) add(rt, g, t0[g], t1[g]);
                        if (LATE && rt + 1 < RT)
                        {
                            asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(dq0[rt + 1]), "+v"(dq1[rt + 1]));
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                }
                else
                {
                    v8bf wa[RT], wb[RT];
#pragma unroll
                    for (int rt = 0; rt < RT; rt++) fields_to_bf16<BITS>(wq[rt], wlo[rt], whi[rt], wa[rt], wb[rt]);
#pragma unroll
                    for (int g = 0; g < MG; g++)
                    {
                        v8bf ya[3], yb[3];
                        v4f t0[RT], t1[RT];
                        split_group(g, ya, yb);
#pragma unroll
                        for (int i = 0; i < 3; i++)
#pragma unroll
                            for (int rt = 0; rt < RT; rt++) product(t0[rt], t1[rt], wa[rt], wb[rt], ya, yb, i);
#pragma unroll
                        for (int rt = 0; rt < RT; rt++) add(rt, g, t0[rt], t1[rt]);
                    }
                }
            }
        }
        WAIT_VMCNT(0); // the surplus loads of the last step must not land on the sums below, nor on the first step again
        if (!F32 || careful) break;
        float nan = 0.f; // (a sum that is none: see split8_bf16x3)
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
#pragma unroll
            for (int g = 0; g < MG; g++)
#pragma unroll
                for (int r = 0; r < 4; r++) nan = acc[rt][g][r] != acc[rt][g][r] ? 1.f : nan;
        if (!__any(nan != 0.f)) break;
    }
    __builtin_amdgcn_s_setprio(0);
    __syncthreads();

    // accumulator r of lane l: weight row (l / 16) * 4 + r of the tile, activation row l % 16 of the group
    float4* red = reinterpret_cast<float4*>(lds_rows);
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int g = 0; g < MG; g++) red[((rt * MG + g) * nwaves + wave) * 64 + lane] = make_float4(acc[rt][g][0], acc[rt][g][1], acc[rt][g][2], acc[rt][g][3]);
    __syncthreads();
    const float* c = mm.c[mat];
    const int bt = mm.bt[mat];
    const float alpha = mm.alpha[mat], beta = mm.beta[mat];
    float* out = mm.out[mat];
    const size_t out_stride = mm.out_stride[mat];
    const bool out_vec = out_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
    for (int p = wave; p < RT * MG; p += nwaves)
    {
        const int rt = p / MG, g = p - rt * MG;
        const int i = g * 16 + m;
        if (i >= M) continue;
        float4 f = red[p * nwaves * 64 + lane];
        const auto add = [&](const float4& o) {
            f.x = add_rn(f.x, o.x);
            f.y = add_rn(f.y, o.y);
            f.z = add_rn(f.z, o.z);
            f.w = add_rn(f.w, o.w);
        };
        constexpr int MOST = rows_waves(BITS, MG, RT, SPLIT, AIN);
        if (nwaves == MOST) // nearly always: all sums requested at once
        {
            float4 o[MOST];
#pragma unroll
            for (int w = 1; w < MOST; w++) o[w] = red[(p * MOST + w) * 64 + lane];
#pragma unroll
            for (int w = 1; w < MOST; w++) add(o[w]);
        }
        else
            for (int w = 1; w < nwaves; w++) add(red[(p * nwaves + w) * 64 + lane]);
        float fr[4] = {f.x, f.y, f.z, f.w};
        const int j0 = (group * RT + rt) * 16 + kg * 4;
        float* to = out + (size_t)(row0 + i) * out_stride + j0;
#pragma unroll
        for (int r = 0; r < 4; r++)
        {
            if (bt >= 0 && j0 + r < N) fr[r] = add_rn(mul_rn(load_c(c, bt, row0 + i, j0 + r, N), beta), fr[r]);
            fr[r] = mul_rn(fr[r], alpha);
        }
        if (out_vec && j0 + 4 <= N)
            *reinterpret_cast<float4*>(to) = make_float4(fr[0], fr[1], fr[2], fr[3]);
        else
        {
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (j0 + r < N) to[r] = fr[r];
        }
    }
}

template<int BITS, bool HALVES, int SPLIT, int MG, int RT, int AIN>
static int launch_one(const void* a, size_t a_stride, int M, int K, int passes, const float* in_scales, BqMulti mm, hipStream_t stream)
{
    const int kblocks = (K + 63) / 64;
    constexpr int PER_WAVE = rows_wave_bytes(BITS, MG, RT, SPLIT, AIN), FIT = rows_waves(BITS, MG, RT, SPLIT, AIN);
    const int nwaves = kblocks < FIT ? kblocks : FIT;
    const size_t lds = (size_t)nwaves * PER_WAVE;
    long long groups = 0;
    for (int i = 0; i < mm.count; i++)
    {
        groups += ((mm.N[i] + 15) / 16 + RT - 1) / RT;
        mm.tile_end[i] = (int)groups;
    }
    const long long blocks = (groups + 7) / 8 * 8 * passes;
    NCNNHIP_REQUIRE(blocks <= 0x7fffffff, "blockquant_rows_kernel: too many workgroups");
    auto kernel = blockquant_rows_kernel<BITS, HALVES, SPLIT, MG, RT, AIN>;
    // more than the 64 KB a kernel gets by default: raised once per device
    static std::atomic<unsigned char> raised[64];
    int device = 0;
    NCNNHIP_CHECK(hipGetDevice(&device));
    if (device < 0 || device >= 64 || !raised[device].load(std::memory_order_acquire))
    {
        NCNNHIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        if (device >= 0 && device < 64) raised[device].store(1, std::memory_order_release);
    }
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(nwaves * 64), lds, stream, a, a_stride, M, K, kblocks, (int)groups, passes, in_scales, mm);
    return launch_status("blockquant_rows_kernel");
}

int launch_blockquant_rows_f16(const uint16_t* a, size_t a_stride, int M, int K, int bits, int block, const BqMulti& mm, hipStream_t stream)
{
    // Groups of activation rows and tiles per workgroup: the cheapest pair under 3.7 us + rounds x K / 4096 x (1.8 MG + 1.6 RT) us (one
    // workgroup per unit, 256 units).  As a forecast that is rough -- off by 13 % in the median and up to half over every pair of MG 1
    // to 4 and RT 1, 2, 3, 4, 6 at N and K 1024 to 27648, 24 to 128 rows, 4 and 8 bits, weights from HBM -- but it ranks well: what it
    // picks took 1 % more than the best pair in the median of those 120 launches, 10 % at most (24 rows of 5120 x 13824 at 4 bits 24.7
    // us with 2 x 2, 1 x 3 22.4; 100 rows of 1024 x 8192 12.1, 2 x 1 11.2).  48 rows of 11008 x 4096 get 3 x 3: 230 workgroups;
    // 3 x 2 are 344, a second round for 88 of them.  Several matrices are counted one by one, as no group has tiles of two: three of 4096 x
    // 4096 are 258 groups of three tiles, not 256, and get 3 x 4 (a decoder layer's seven matrices at 4 bits, 48 rows, 76.9 -> 68.2 us;
    // groups across matrices took 67.2 but cost every other launch up to a microsecond in looking them up).
    const int rows16 = (M + 15) / 16;
    int mg = 4, rt = 4;
    double best = 0.0;
    for (int g = 1; g <= 4; g++)
        for (const int r : {1, 2, 3, 4, 6})
        {
            long long wgs = 0;
            for (int i = 0; i < mm.count; i++) wgs += ((mm.N[i] + 15) / 16 + r - 1) / r; // no group has tiles of two matrices
            wgs *= (rows16 + g - 1) / g;
            const double cost = (double)((wgs + 255) / 256) * (1.8 * g + 1.6 * r);
            if (best == 0.0 || cost < best) best = cost, mg = g, rt = r;
        }
    const int passes = (rows16 + mg - 1) / mg;
#define ONE(BITS_, HALVES_, SPLIT_, MG_, RT_) return launch_one<BITS_, HALVES_, SPLIT_, MG_, RT_, 2>(a, a_stride, M, K, passes, nullptr, mm, stream)
#define ONE_RT(BITS_, HALVES_, SPLIT_, MG_)              \
    do                                                   \
    {                                                    \
        if (rt == 1) ONE(BITS_, HALVES_, SPLIT_, MG_, 1); \
        if (rt == 2) ONE(BITS_, HALVES_, SPLIT_, MG_, 2); \
        if (rt == 3) ONE(BITS_, HALVES_, SPLIT_, MG_, 3); \
        if (rt == 4) ONE(BITS_, HALVES_, SPLIT_, MG_, 4); \
        ONE(BITS_, HALVES_, SPLIT_, MG_, 6);             \
    } while (0)
#define ONE_MG(BITS_, HALVES_, SPLIT_)            \
    do                                            \
    {                                             \
        if (mg == 1) ONE_RT(BITS_, HALVES_, SPLIT_, 1); \
        if (mg == 2) ONE_RT(BITS_, HALVES_, SPLIT_, 2); \
        if (mg == 3) ONE_RT(BITS_, HALVES_, SPLIT_, 3); \
        ONE_RT(BITS_, HALVES_, SPLIT_, 4);        \
    } while (0)
    const bool split = block == 32;
    if (!halves_layout(bits, block)) ONE_MG(8, false, 0);
    if (bits == 8) ONE_MG(8, true, 1); // blocks of 32 only
    if (bits == 6 && split) ONE_MG(6, true, 1);
    if (bits == 6) ONE_MG(6, true, 0);
    if (split) ONE_MG(4, true, 1);
    ONE_MG(4, true, 0);
#undef ONE_MG
#undef ONE_RT
#undef ONE
}

// fp32 rows: groups of activation rows and tiles per workgroup, the cheapest pair under rounds x (2.3 + 0.7 MG RT + K / 4096 x (4 + 2.2 MG +
// 1.4 MG RT)) us, the form of 90 measured pairs at 8 bits (four groups leave room for 4 or 5 wavefronts and were not better anywhere).  The grid's
// padding to 8 groups counts: 81 groups in 3 passes are 264 workgroups, a second round (37 rows of 5154 x 768 13.0 us with 1 x 4, 8.8
// with 2 x 3).  Several matrices are counted one by one, as for fp16 rows.
double blockquant_rows_f32_us(int M, int K, const int* N, int count, int* mg, int* rt)
{
    const int rows16 = (M + 15) / 16;
    double best = 0.0;
    for (int g = 1; g <= 2; g++)
        for (int r = 1; r <= 4; r++)
        {
            long long wgs = 0;
            for (int i = 0; i < count; i++) wgs += ((N[i] + 15) / 16 + r - 1) / r;
            wgs = (wgs + 7) / 8 * 8 * ((rows16 + g - 1) / g);
            const double us = (double)((wgs + 255) / 256) * (2.3 + 0.7 * g * r + K / 4096.0 * (4.0 + 2.2 * g + 1.4 * g * r));
            if (best == 0.0 || us < best) best = us, *mg = g, *rt = r;
        }
    return best;
}

int launch_blockquant_rows_f32(const float* a, size_t a_stride, int M, int K, int bits, int block, const float* in_scales, const BqMulti& mm, hipStream_t stream)
{
    int mg = 1, rt = 1;
    blockquant_rows_f32_us(M, K, mm.N, mm.count, &mg, &rt);
    const int passes = ((M + 15) / 16 + mg - 1) / mg;
#define ONE(BITS_, HALVES_, SPLIT_, MG_, RT_) return launch_one<BITS_, HALVES_, SPLIT_, MG_, RT_, 4>(a, a_stride, M, K, passes, in_scales, mm, stream)
#define ONE_RT(BITS_, HALVES_, SPLIT_, MG_)              \
    do                                                   \
    {                                                    \
        if (rt == 1) ONE(BITS_, HALVES_, SPLIT_, MG_, 1); \
        if (rt == 2) ONE(BITS_, HALVES_, SPLIT_, MG_, 2); \
        if (rt == 3) ONE(BITS_, HALVES_, SPLIT_, MG_, 3); \
        ONE(BITS_, HALVES_, SPLIT_, MG_, 4);             \
    } while (0)
#define ONE_MG(BITS_, HALVES_, SPLIT_)            \
    do                                            \
    {                                             \
        if (mg == 1) ONE_RT(BITS_, HALVES_, SPLIT_, 1); \
        ONE_RT(BITS_, HALVES_, SPLIT_, 2);        \
    } while (0)
    const bool split = block == 32;
    if (!halves_layout(bits, block)) ONE_MG(8, false, 0);
    if (bits == 8) ONE_MG(8, true, 1); // blocks of 32 only
    if (bits == 6 && split) ONE_MG(6, true, 1);
    if (bits == 6) ONE_MG(6, true, 0);
    if (split) ONE_MG(4, true, 1);
    ONE_MG(4, true, 0);
#undef ONE_MG
#undef ONE_RT
#undef ONE
}

} // namespace ncnnhip
