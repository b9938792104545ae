// Block-quantised Gemm on many fp16 activation rows (from 5, by weights: many_rows_f16): every weight is read once for up to 64 rows.
//
// The few-row kernels (blockquant.hip) multiply 16 rows per pass over the weights; 48 rows were three passes of a launch each.
// Here a workgroup owns RT tiles of 16 weight rows and MG groups of 16 activation rows and deals the K steps of 64 out to its
// wavefronts, each a run of its own.  A wavefront streams what a step needs -- MG x 16 rows of 128 bytes, its RT tiles
// and their descales -- from global memory straight into LDS, into a ring of two stages that belongs to it alone: no barrier and
// no other wavefront stands in its way, and the eight of a workgroup keep about 80 KB in flight on a compute unit.  The sums
// of the wavefronts meet in LDS at the end.
//
// What bounds it is not the weights but the activations: every workgroup reads all M x K of them (393 KB for 48 rows of 4096)
// through its unit's L1, so MG and RT balance re-reading them against idle units (launch_blockquant_rows_f16).
// us per launch, 16 rows per pass -> here, weights from HBM, 4 bits in blocks of 64: 4096 x 4096 24 rows 11.9 -> 8.9, 48 rows 18.4 -> 10.8,
// 128 rows 45.9 -> 14.6; 11008 x 4096 48 rows 37.3 -> 16.8; 4096 x 11008 48 rows 102 -> 21.5; 8 bits 48 rows 4096 x 4096 20.0 -> 11.3,
// 11008 x 4096 42.6 -> 19.1, 4096 x 11008 48.0 -> 23.4.
// A lane must fetch along a row (eight lanes = one 128-byte line) and read in operand order (lane = row), so the chunks of a row
// are swizzled on the source side: chunk c of row r lands at position c ^ ((r / 2) % 8), conflict-free both ways.
#include <atomic>

#include "blockquant.h"

#define AS1 __attribute__((address_space(1)))
#define AS3 __attribute__((address_space(3)))

namespace ncnnhip {

// s_waitcnt immediate that waits for vmcnt <= n only (gfx9 encoding)
#define WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(0x0F70 | ((n) & 15) | ((((n) >> 4) & 3) << 14))

constexpr int ROWS_MAX_WAVES = 8;

constexpr int rows_stage_bytes(int bits, int mg, int rt, int split)
{
    return mg * 2048 + rt * 128 * bits + rt * (64 << split);
}
template<int BITS, bool HALVES, int SPLIT, int MG, int RT>
__global__ __launch_bounds__(ROWS_MAX_WAVES * 64) void blockquant_rows_f16_kernel(const __half* __restrict__ a, size_t a_stride, int M_total, int K, int kblocks,
                                                                                  int groups, int passes, BqMulti mm)
{
    static_assert(HALVES || (BITS == 8 && SPLIT == 0), "4- and 6-bit fields and blocks of 32 come in the halves layout");
    constexpr int STEP_BYTES = 128 * BITS;   // one tile's weights for a step
    constexpr int DPER = 4 << SPLIT;         // its descales, in float4
    constexpr int W_OFF = MG * 2048, D_OFF = W_OFF + RT * STEP_BYTES;
    constexpr int STAGE = rows_stage_bytes(BITS, MG, RT, SPLIT);
    constexpr int LOADS = MG * 2 + RT + 1;
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
    while (mat + 1 < mm.count && group >= mm.tile_end[mat]) mat++;
    group -= mat ? mm.tile_end[mat - 1] : 0;
    const int N = mm.N[mat], ntiles = (N + 15) >> 4;
    const int M = M_total - row0 < MG * 16 ? M_total - row0 : MG * 16;

    // this wavefront's K steps
    const int step0 = (int)((long long)kblocks * wave / nwaves), steps = (int)((long long)kblocks * (wave + 1) / nwaves) - step0;
    const int ragged = (K & 63) ? kblocks - 1 - step0 : -1; // the step K ends in (the last wavefront's; beyond the others' steps)

    // sources.  Activations: load i brings rows i * 8 .. + 8 of the pass, lane l row l / 8 and the chunk that belongs at position l % 8
    const __half* arow[MG * 2];
#pragma unroll
    for (int i = 0; i < MG * 2; i++)
    {
        const int r = i * 8 + (lane >> 3);
        arow[i] = a + (size_t)(row0 + (r < M ? r : M - 1)) * a_stride;
    }
    const int chunk0 = (lane & 7) ^ ((lane >> 4) & 7); // even i; odd i: chunk0 ^ 4
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
        const int k0 = (step0 + s) * 64 + chunk0 * 8, k1 = (step0 + s) * 64 + (chunk0 ^ 4) * 8;
        const int c0 = k0 < K ? k0 : 0, c1 = k1 < K ? k1 : 0; // K % 16 == 0: a chunk is all in or all out
#pragma unroll
        for (int i = 0; i < MG * 2; i++)
            __builtin_amdgcn_global_load_lds((const AS1 void*)(arow[i] + (i & 1 ? c1 : c0)), (AS3 void*)(st + i * 1024), 16, 0, 0);
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
            if (lane < STEP_BYTES / 16)
                __builtin_amdgcn_global_load_lds((const AS1 void*)(wsrc[rt] + (size_t)s * STEP_BYTES), (AS3 void*)(st + W_OFF + rt * STEP_BYTES), 16, 0, 0);
        if (lane < RT * DPER) __builtin_amdgcn_global_load_lds((const AS1 void*)(dsrc + (size_t)s * DPER), (AS3 void*)(st + D_OFF), 16, 0, 0);
    };

    v4f acc[RT][MG];
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int g = 0; g < MG; g++) acc[rt][g] = v4f{0.f, 0.f, 0.f, 0.f};

    const int sw = (m >> 1) & 7;
    const unsigned base = (unsigned)(uintptr_t)(AS3 unsigned char*)ring;
    const unsigned rd_a = base + m * 128 + (((HALVES ? kg : 2 * kg) ^ sw) << 4);
    const unsigned rd_b = base + m * 128 + (((HALVES ? 4 + kg : 2 * kg + 1) ^ sw) << 4);
    const unsigned rd_w = base + W_OFF + lane * (BITS == 8 ? 16 : 8), rd_w3 = base + W_OFF + 512 + lane * 4;
    const unsigned rd_d = base + D_OFF + kg * 16;

    issue(0, 0);
    for (int s = 0; s < steps; s++)
    {
        const unsigned at = (unsigned)((s & 1) * STAGE);
        // the stage multiplied in the turn before has been read (its reads were waited for): the next loads go there
        issue(s + 1 < steps ? s + 1 : s, (s + 1) & 1);
        WAIT_VMCNT(LOADS);
        asm volatile("" ::: "memory");
        if (s == ragged)
        {
            // zeros in place of the chunks beyond K: their weights are zero, but zero times an infinity is not
            const v4i_bq zeros = {0, 0, 0, 0};
            const int k0 = (step0 + s) * 64 + chunk0 * 8, k1 = (step0 + s) * 64 + (chunk0 ^ 4) * 8;
#pragma unroll
            for (int i = 0; i < MG * 2; i++)
                if ((i & 1 ? k1 : k0) >= K) asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(base + at + lane * 16), "v"(zeros), "n"(i * 1024) : "memory");
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
            asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dq0[rt]) : "v"(rd_d + at), "n"(rt * DPER * 16));
            if (SPLIT) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dq1[rt]) : "v"(rd_d + at), "n"(rt * DPER * 16 + 64));
        }
        union Act
        {
            v4i_bq i4;
            v8h h;
        };
        Act xa[MG], xb[MG];
#pragma unroll
        for (int g = 0; g < MG; g++)
        {
            asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(xa[g].i4) : "v"(rd_a + at), "n"(g * 2048));
            asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(xb[g].i4) : "v"(rd_b + at), "n"(g * 2048));
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
        {
            if (BITS == 8)
                asm volatile("" : "+v"(wq[rt]));
            else
                asm volatile("" : "+v"(wlo[rt]));
            if (BITS == 6) asm volatile("" : "+v"(whi[rt]));
            asm volatile("" : "+v"(dq0[rt]));
            if (SPLIT) asm volatile("" : "+v"(dq1[rt]));
        }
#pragma unroll
        for (int g = 0; g < MG; g++) asm volatile("" : "+v"(xa[g].i4), "+v"(xb[g].i4));
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
        {
            v8h wa, wb;
            if (BITS == 8)
            {
                wa = bytes_to_halves(wq[rt][0], wq[rt][1]);
                wb = bytes_to_halves(wq[rt][2], wq[rt][3]);
            }
            else if (BITS == 4)
            {
                wa = nibbles_to_halves((unsigned)wlo[rt][0]);
                wb = nibbles_to_halves((unsigned)wlo[rt][1]);
            }
            else
                sixbit_to_halves((unsigned)wlo[rt][0], (unsigned)wlo[rt][1], (unsigned)whi[rt], wa, wb);
            const v4f zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int g = 0; g < MG; g++)
            {
                v4f t0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(wa, xa[g].h, zero, 0, 0, 0);
                const v4f t1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(wb, xb[g].h, SPLIT ? zero : t0, 0, 0, 0);
                if (!SPLIT) t0 = t1;
#pragma unroll
                for (int r = 0; r < 4; r++)
                {
                    acc[rt][g][r] = fmaf(t0[r], __int_as_float(dq0[rt][r]), acc[rt][g][r]);
                    if (SPLIT) acc[rt][g][r] = fmaf(t1[r], __int_as_float(dq1[rt][r]), acc[rt][g][r]);
                }
            }
        }
    }
    WAIT_VMCNT(0); // the surplus loads of the last step must not land on the sums below
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
    for (int p = wave; p < RT * MG; p += nwaves)
    {
        const int rt = p / MG, g = p - rt * MG;
        const int i = g * 16 + m;
        if (i >= M) continue;
        float4 f = red[p * nwaves * 64 + lane];
        for (int w = 1; w < nwaves; w++)
        {
            const float4 o = red[(p * nwaves + w) * 64 + lane];
            f.x = add_rn(f.x, o.x);
            f.y = add_rn(f.y, o.y);
            f.z = add_rn(f.z, o.z);
            f.w = add_rn(f.w, o.w);
        }
        const float fr[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
        for (int r = 0; r < 4; r++)
        {
            const int j = (group * RT + rt) * 16 + kg * 4 + r;
            if (j < N)
            {
                float v = fr[r];
                if (bt >= 0) v = add_rn(mul_rn(load_c(c, bt, row0 + i, j, N), beta), v);
                out[(size_t)(row0 + i) * out_stride + j] = mul_rn(v, alpha);
            }
        }
    }
}

template<int BITS, bool HALVES, int SPLIT, int MG, int RT>
static int launch_one(const __half* a, size_t a_stride, int M, int K, int passes, BqMulti mm, hipStream_t stream)
{
    const int kblocks = (K + 63) / 64;
    constexpr int STAGE = rows_stage_bytes(BITS, MG, RT, SPLIT);
    constexpr int PER_WAVE = 2 * STAGE > RT * MG * 1024 ? 2 * STAGE : RT * MG * 1024; // its ring, later its sums
    constexpr int FIT = 160 * 1024 / PER_WAVE < ROWS_MAX_WAVES ? 160 * 1024 / PER_WAVE : ROWS_MAX_WAVES;
    const int nwaves = kblocks < FIT ? kblocks : FIT;
    const size_t lds = (size_t)nwaves * PER_WAVE;
    long long groups = 0;
    for (int i = 0; i < mm.count; i++)
    {
        groups += ((mm.N[i] + 15) / 16 + RT - 1) / RT;
        mm.tile_end[i] = (int)groups;
    }
    const long long blocks = (groups + 7) / 8 * 8 * passes;
    NCNNHIP_REQUIRE(blocks <= 0x7fffffff, "blockquant_rows_f16_kernel: too many workgroups");
    auto kernel = blockquant_rows_f16_kernel<BITS, HALVES, SPLIT, MG, RT>;
    // more than the 64 KB a kernel gets by default: raised once per device
    static std::atomic<unsigned char> raised[64];
    int device = 0;
    NCNNHIP_CHECK(hipGetDevice(&device));
    if (device < 0 || device >= 64 || !raised[device].load(std::memory_order_acquire))
    {
        NCNNHIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        if (device >= 0 && device < 64) raised[device].store(1, std::memory_order_release);
    }
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(nwaves * 64), lds, stream, a, a_stride, M, K, kblocks, (int)groups, passes, mm);
    return launch_status("blockquant_rows_f16_kernel");
}

int launch_blockquant_rows_f16(const uint16_t* a_, size_t a_stride, int M, int K, int bits, int block, const BqMulti& mm, hipStream_t stream)
{
    const __half* a = reinterpret_cast<const __half*>(a_);
    // Groups of activation rows and tiles per workgroup: the cheapest pair under 3.7 us + rounds x K / 4096 x (1.8 MG + 1.6 RT) us (one
    // workgroup per unit, 256 units).  As a forecast that is rough -- off by 13 % in the median and up to half over every pair of MG 1
    // to 4 and RT 1, 2, 3, 4, 6 at N and K 1024 to 27648, 24 to 128 rows, 4 and 8 bits, weights from HBM -- but it ranks well: what it
    // picks took 1 % more than the best pair in the median of those 120 launches, 10 % at most (24 rows of 5120 x 13824 at 4 bits 24.7
    // us with 2 x 2, 1 x 3 22.4; 100 rows of 1024 x 8192 12.1, 2 x 1 11.2).  48 rows of 11008 x 4096 get 3 x 3: 230 workgroups;
    // 3 x 2 are 344, a second round for 88 of them.
    const int rows16 = (M + 15) / 16;
    long long tiles = 0;
    for (int i = 0; i < mm.count; i++) tiles += (mm.N[i] + 15) / 16;
    int mg = 4, rt = 4;
    double best = 0.0;
    for (int g = 1; g <= 4; g++)
        for (const int r : {1, 2, 3, 4, 6})
        {
            const long long wgs = ((tiles + r - 1) / r) * ((rows16 + g - 1) / g);
            const double cost = (double)((wgs + 255) / 256) * (1.8 * g + 1.6 * r);
            if (best == 0.0 || cost < best) best = cost, mg = g, rt = r;
        }
    const int passes = (rows16 + mg - 1) / mg;
#define ONE(BITS_, HALVES_, SPLIT_, MG_, RT_) return launch_one<BITS_, HALVES_, SPLIT_, MG_, RT_>(a, a_stride, M, K, passes, mm, stream)
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

} // namespace ncnnhip
