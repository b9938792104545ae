// Block-quantised Gemm on many rows of fp32 activations (prefill, attention projections), weights in blocks of 64 or 128: the activations
// are split into three bf16 numbers by a pass of its own, then a workgroup multiplies 64 of their rows with 128 weight rows on
// v_mfma_f32_32x32x16_bf16.
//
// A wavefront multiplies 64 activation rows with 64 weight rows and a workgroup holds four groups of two, each with a quarter of K: a weight
// is converted to bf16 once for 64 rows (with 32, as blockquant.hip's kernels have it, the vector unit is as busy as the matrix cores), and
// 256 tiles of 64 x 128, a prefill of 512 rows of 4096, still put two wavefronts on every SIMD.
// Bound by the matrix cores' issue and the clock, 1.8 GHz on all units: half a K step takes a wavefront about 1100 cycles of multiplying for
// 768 of matrix-core time (the rest: nine loads, 14 of their cycles each not hidden, and the conversions), and its neighbour reads meanwhile.
// us with the split pass (7 at 512 x 4096), 8 bits in blocks of 64, blockquant.hip's kernels -> here: 512 x 4096 x 4096 78 -> 65, 512 x 4096 x 11008
// 178 -> 139, 512 x 11008 x 4096 162 -> 150, 333 x 4096 x 4096 66 -> 50, 1500 x 1024 x 1024 29.5 -> 24.6; 4 bits 512 x 4096 x 4096 87 -> 60.
// Error against 64 bits 1.26e-7 for 1.44e-7.  (Weights and loads all before the products: 70; activations requested half a stage later, where the
// wavefront does not multiply: 74; two groups and two workgroups to a unit: 68, and 4 % quicker only on many rounds.)
#include <atomic>

#include "blockquant.h"

#define AS1 __attribute__((address_space(1)))
#define AS3 __attribute__((address_space(3)))
#define WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(0x0F70 | ((n) & 15) | ((((n) >> 4) & 3) << 14))

namespace ncnnhip {

typedef float v16f_bq __attribute__((ext_vector_type(16)));

// ---- the activations in operand order ----
// A stage is half a K step: of the 16-byte pieces the packed weights keep for four K groups (two chunks of 8 each) those of groups 2 h and
// 2 h + 1.  [row block of 64][K step][h] [32-row group][chunk c of the piece][part] 64 lanes x 16 bytes: lane = row l % 32, K group 2 h + l / 32.
// Rows beyond M and K beyond the last are zeros.  One workgroup: 64 rows x two K steps.
template<bool HALVES>
__global__ __launch_bounds__(256) void blockquant_split_tiles_kernel(const float* __restrict__ a, size_t a_stride, int M, int K, int kblocks,
                                                                     const float* __restrict__ in_scales, uint4* __restrict__ frags)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l32 = lane & 31, hh = lane >> 5;
    const int h = wave >> 1, c = wave & 1;
    const int chunk = HALVES ? 2 * h + hh + 4 * c : 2 * (2 * h + hh) + c;
    float x[4][8];
#pragma unroll
    for (int u = 0; u < 4; u++)
    {
        const int kb = blockIdx.x * 2 + (u >> 1), row = blockIdx.y * 64 + (u & 1) * 32 + l32, k = kb * 64 + chunk * 8;
        const bool inside = row < M && k < K; // K % 16 == 0: a chunk of 8 is all in or all out
        const float* p = a + (inside ? (size_t)row * a_stride + k : (size_t)0);
#pragma unroll
        for (int j = 0; j < 8; j++) x[u][j] = p[j]; // a valid address either way (K >= 16)
        if (!inside)
        {
#pragma unroll
            for (int j = 0; j < 8; j++) x[u][j] = 0.f;
        }
        else if (in_scales)
        {
#pragma unroll
            for (int j = 0; j < 8; j++) x[u][j] = mul_rn(x[u][j], in_scales[k + j]);
        }
    }
#pragma unroll
    for (int u = 0; u < 4; u++)
    {
        const int kb = blockIdx.x * 2 + (u >> 1);
        if (kb >= kblocks) break;
        unsigned pl[3][4];
#pragma unroll
        for (int e = 0; e < 4; e++)
        {
            unsigned part[2][3];
#pragma unroll
            for (int o = 0; o < 2; o++) split_bf16x3(x[u][2 * e + o], part[o][0], part[o][1], part[o][2]);
#pragma unroll
            for (int p = 0; p < 3; p++) pl[p][e] = (part[0][p] >> 16) | part[1][p];
        }
        uint4* to = frags + ((((size_t)blockIdx.y * kblocks + kb) * 2 + h) * 12 + ((u & 1) * 2 + c) * 3) * 64 + lane;
#pragma unroll
        for (int p = 0; p < 3; p++) to[p * 64] = make_uint4(pl[p][0], pl[p][1], pl[p][2], pl[p][3]);
    }
}

constexpr int TILES_STAGE = 12 * 1024; // bytes of activations
constexpr int tiles_weight_bytes(int bits) { return 8 * 64 * bits + 512; }
constexpr int KG = 4; // groups of two wavefronts
constexpr int tiles_lds_bytes(int bits) { return KG * (2 * TILES_STAGE + 3 * tiles_weight_bytes(bits)); } // (more than the 96 KB the sums take later)

// Each group has a ring of its own for two stages of activations (12 KB, read by both wavefronts) and three of weights and descales (read by
// the wavefront that fetched them, a stage ahead, and converted while it multiplies), filled straight from global memory as soon as
// the operands are in registers.  The last two groups run half a stage behind the first two, their neighbours on the same SIMDs: one
// reads while the other multiplies.
template<int BITS>
__global__ __launch_bounds__(KG * 128) void blockquant_tiles_kernel(const uint4* __restrict__ frags, int M, int N, int kblocks, int ntiles,
                                                                   const unsigned char* __restrict__ wpk, const float4* __restrict__ dpk, const float* __restrict__ c,
                                                                   int bt, float alpha, float beta, float* __restrict__ out, size_t out_stride)
{
    constexpr int LOADS = 6 + (BITS == 4 ? 1 : BITS == 8 ? 2 : 3) + 1; // per wavefront and stage
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
    const char* const abase = reinterpret_cast<const char*>(frags + ((size_t)blockIdx.y * kblocks * 24 + ww * 6) * 64);
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
    // load i of a stage: 6 of activations (of half h of K step `at`; h is also their slot), the others of weights (of a later stage)
    const auto load_activations = [&](int at, int h, int i) {
        const char* from = abase + (size_t)((at < last ? at : last) * 2 + h) * TILES_STAGE;
        __builtin_amdgcn_global_load_lds((const AS1 void*)(from + (unsigned)(lane * 16 + i * 1024)), (AS3 void*)(mine + h * TILES_STAGE + (ww * 6 + i) * 1024), 16, 0, 0);
    };
    const auto load_weights = [&](int at, int h, int slot, int i) {
        const int kb = at < last ? at : last;
        unsigned char* st = mine + 2 * TILES_STAGE + slot * WSTAGE;
        const char* from = wbase + (size_t)kb * STEP_BYTES + h * (BITS == 8 ? 512 : 256);
        if (i == LOADS - 7)
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
        for (int i = 0; i < 6; i++) load_activations(at, h, i);
    };
    const auto issue_weights = [&](int at, int h, int slot) {
#pragma unroll
        for (int i = 0; i < LOADS - 6; i++) load_weights(at, h, slot, i);
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
    const auto convert = [&](v8bf (&w)[2][2], int part) { // [32 weight rows][chunk], in four parts
        const int g = part >> 1, ch = part & 1;
        if constexpr (BITS == 8)
            w[g][ch] = bytes_to_bf16((unsigned)wq[g][2 * ch], (unsigned)wq[g][2 * ch + 1]);
        else if constexpr (BITS == 4)
            w[g][ch] = nibbles_to_bf16((unsigned)wlo[g][ch]);
        else if (ch == 0)
            sixbit_to_bf16((unsigned)wlo[g][0], (unsigned)wlo[g][1], (unsigned)whi[g], w[g][0], w[g][1]);
    };

    v8bf w[2][2];
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
            v8bf b;
        };
        Act y[12];
#pragma unroll
        for (int i = 0; i < 12; i++) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(y[i].i4) : "v"(a_at), "n"(h * TILES_STAGE + i * 1024));
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
        for (int i = 0; i < 12; i++) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(y[i].i4));
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
        v8bf wn[2][2]; // the next stage's
        // six rounds of four products; the loads and the conversions spread over them
#pragma unroll
        for (int c = 0; c < 6; c++)
        {
            const int ch = c / 3, p = c % 3;
#pragma unroll
            for (int i = c * LOADS / 6; i < (c + 1) * LOADS / 6; i++)
            {
                if (i < 6)
                    load_activations(kb + 1, h, i);
                else
                    load_weights(h == 0 ? kb + 1 : kb + 2, h ^ 1, slot, i - 6);
            }
#pragma unroll
            for (int q = 0; q < 4; q++) t[q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(y[((q >> 1) * 2 + ch) * 3 + p].b, w[q & 1][ch], t[q], 0, 0, 0);
            if (c < 4) convert(wn, c);
#pragma unroll
            for (int q = 0; q < 4; q++)
            {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (q < (c + 1) * LOADS / 6 - c * LOADS / 6) __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
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
        const int j = (tile0 + 2 * (q & 1)) * 16 + l32;
        if (j >= N) continue;
#pragma unroll
        for (int r = 0; r < 16; r++)
        {
            const int i = row0 + (q >> 1) * 32 + 8 * (r >> 2) + 4 * hh + (r & 3);
            if (i < M)
            {
                float v = acc[q][r];
                if (bt >= 0) v = add_rn(mul_rn(load_c(c, bt, i, j, N), beta), v);
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
    const dim3 sgrid((unsigned)((kblocks + 1) / 2), (unsigned)blocks), grid((unsigned)((ntiles + 7) / 8), (unsigned)blocks);
    if (bits == 8)
        hipLaunchKernelGGL(blockquant_split_tiles_kernel<false>, sgrid, dim3(256), 0, st, a, a_stride, M, K, kblocks, in_scales, frags);
    else
        hipLaunchKernelGGL(blockquant_split_tiles_kernel<true>, sgrid, dim3(256), 0, st, a, a_stride, M, K, kblocks, in_scales, frags);
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
        hipLaunchKernelGGL(kernel, grid, dim3(KG * 128), tiles_lds_bytes(BITS_), st, frags, M, N, kblocks, ntiles, wpk, dpk, c, bt, alpha, beta, out,      \
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
