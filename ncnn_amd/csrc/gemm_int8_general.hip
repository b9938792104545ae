// int8 Gemm and InnerProduct of any shape, stride and alignment on the gfx950 matrix cores.
//
// The ring kernels of gemm_int8_pipelined.hip copy global memory straight into LDS and so need rows on 16-byte boundaries and
// whole K steps.  Here an operand row may start at any byte and K may end anywhere: a lane fetches 16 bytes of a row into
// registers (an unaligned global load; it costs what the cache lines it touches cost), two or three K steps ahead, and
// writes them to LDS when the step before is being multiplied.  K past the end is zero in both operands, rows past the end
// repeat the last one and are never stored.
//
// A workgroup is four wavefronts, 2 x 2, on a BM x BN tile; a K step is 128 bytes of every row.  LDS holds two steps; row r
// keeps its eight 16-byte chunks at positions c ^ ((r >> 1) & 7), so that any 16 consecutive rows read at one K offset meet
// 16 different bank groups.  One barrier per step: the buffer that step t + 1 is written into was last read in step t - 1.
// Bound by latency at the sizes it is for (a few hundred tiles of 64 x 64): 1501 x 1000 x 2008 168 us with the byte gathers
// of the kernel before this one.
#include "conv_nhwc.h"
#include "epilogues.h"
#include "gemm_int8_general.h"

namespace ncnnhip {

constexpr int KSTEP = 128;

// ---- epilogues: one value per tile row (made once, kept in LDS), a scale and an addend per column (made once per lane)
// PLAIN: C none or per column, row-major output, no accumulator dump
template<bool PLAIN>
struct TileGemm
{
    GemmEpilogue e;
    __device__ __forceinline__ float row_value(int i) const
    {
        return e.per_col ? div_rn(1.f, e.a_scales[i]) : div_rn(1.f, mul_rn(e.a_scales[i], e.b_scales[0]));
    }
    __device__ __forceinline__ void column(int j, float& scale, float& add) const
    {
        scale = e.per_col ? div_rn(1.f, e.b_scales[j]) : 1.f;
        add = e.bt == 4 ? mul_rn(e.c[j], e.beta) : e.bt == 0 ? mul_rn(e.c[0], e.beta) : 0.f;
    }
    __device__ __forceinline__ void store(int i, int j, int acc, float row, float scale, float add) const
    {
        float f = mul_rn((float)acc, row);
        if (e.per_col) f = mul_rn(f, scale);
        if (PLAIN)
        {
            if (e.bt >= 0) f = add_rn(f, add);
            e.out[(size_t)i * e.out_stride + j] = mul_rn(f, e.alpha);
            return;
        }
        if (e.acc_out) e.acc_out[(size_t)i * e.N + j] = acc;
        if (e.bt == 0 || e.bt == 4)
            f = add_rn(f, add);
        else if (e.bt == 1 || e.bt == 2)
            f = add_rn(f, mul_rn(e.c[i], e.beta));
        else if (e.bt == 3)
            f = add_rn(f, mul_rn(e.c[(size_t)i * e.N + j], e.beta));
        f = mul_rn(f, e.alpha);
        e.out[e.transpose ? (size_t)j * e.out_stride + i : (size_t)i * e.out_stride + j] = f;
    }
};

// InnerProduct: rows are input rows, columns are output channels
struct TileFc
{
    FcEpilogue e;
    __device__ __forceinline__ float row_value(int) const
    {
        return 0.f;
    }
    __device__ __forceinline__ void column(int j, float& scale, float& add) const
    {
        scale = e.scale_in[j];
        add = e.bias ? e.bias[j] : -0.f; // x + -0 is x for every x
    }
    __device__ __forceinline__ void store(int i, int j, int acc, float, float scale, float add) const
    {
        if (e.acc_out) e.acc_out[(size_t)i * e.num_output + j] = acc;
        e.out[(size_t)i * e.out_stride + j] = apply_activation(add_rn(mul_rn((float)acc, scale), add), e.act);
    }
};

// KG groups of four wavefronts share a tile: group g multiplies the K steps g, g + KG, ... through LDS buffers of its own, and the
// groups' sums meet in LDS at the end (integers: any order gives the same).
constexpr int AHEAD = 2; // K steps requested before the one that is being written to LDS (three and four: no faster)
template<int BM, int BN, int KG, typename Epilogue>
__global__ __launch_bounds__(256 * KG) void gemm_int8_general_kernel(const int8_t* __restrict__ A, size_t lda, const int8_t* __restrict__ B, size_t ldb, int M, int N, int K,
                                                                int tiles_m, int tiles_n, Epilogue epi)
{
    constexpr int TM = BM / 64, TN = BN / 64;     // 32 x 32 blocks per wavefront
    constexpr int LA = BM / 32, LB = BN / 32;     // 16-byte loads per thread and operand: 32 rows of 8 chunks at a time
    constexpr int STEP_BYTES = (BM + BN) * KSTEP;
    static_assert(KG == 1 || BM * BN * 4 <= 2 * STEP_BYTES, "the sums of a group fit its buffers");
    __shared__ __attribute__((aligned(16))) int8_t smem_all[KG * 2 * STEP_BYTES];
    __shared__ float row_value[BM];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3);
    const int kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    int8_t* smem = smem_all + kg * 2 * STEP_BYTES;
    const int wm = wave >> 1, wn = wave & 1, l32 = lane & 31, lhi = lane >> 5;

    // workgroups are dealt to the 8 dies in turn: each die takes a run of tiles that share rows of A and B in its own L2
    const int T = tiles_m * tiles_n;
    const int die = blockIdx.x & 7, per_die = T >> 3, more = T & 7;
    const int tile = die * per_die + (die < more ? die : more) + (int)(blockIdx.x >> 3);
    constexpr int GM = 4;
    const int group = tile / (GM * tiles_n);
    const int rows_of_group = tiles_m - group * GM < GM ? tiles_m - group * GM : GM;
    const int in_group = tile - group * GM * tiles_n;
    const int row0 = (group * GM + in_group % rows_of_group) * BM, col0 = in_group / rows_of_group * BN;

    const int ld_row = (threadIdx.x & 255) >> 3, ld_chunk = threadIdx.x & 7;
    const int8_t* pa[LA];
    const int8_t* pb[LB];
    int wr_a[LA], wr_b[LB];
#pragma unroll
    for (int i = 0; i < LA; i++)
    {
        const int r = i * 32 + ld_row;
        pa[i] = A + (size_t)(row0 + r < M ? row0 + r : M - 1) * lda;
        wr_a[i] = r * KSTEP + ((ld_chunk ^ (r >> 1)) & 7) * 16;
    }
#pragma unroll
    for (int i = 0; i < LB; i++)
    {
        const int r = i * 32 + ld_row;
        pb[i] = B + (size_t)(col0 + r < N ? col0 + r : N - 1) * ldb;
        wr_b[i] = BM * KSTEP + r * KSTEP + ((ld_chunk ^ (r >> 1)) & 7) * 16;
    }
    if (threadIdx.x < BM) row_value[threadIdx.x] = row0 + (int)threadIdx.x < M ? epi.row_value(row0 + threadIdx.x) : 0.f;

    // whole steps come from memory as they are; what is left of K (tail > 0 bytes) is requested first and waits in registers
    const int whole_all = K / KSTEP;
    const int tail = whole_all % KG == kg ? K - whole_all * KSTEP : 0; // the group whose turn it would be
    const int whole = (whole_all + KG - 1 - kg) / KG;                  // whole steps of this group
    const int turns = (whole_all + KG - 1) / KG;                       // of the group with the most
    v4i ra[AHEAD][LA], rb[AHEAD][LB], ta[LA], tb[LB];
    const int tail_k = whole_all * KSTEP + ld_chunk * 16, tail_drop = tail_k + 16 - K; // bytes of this lane's chunk beyond K
    if (tail)
    {
        const int k = tail_drop > 0 ? K - 16 : tail_k;
#pragma unroll
        for (int i = 0; i < LA; i++) ta[i] = load16(pa[i] + k);
#pragma unroll
        for (int i = 0; i < LB; i++) tb[i] = load16(pb[i] + k);
    }
    // No branch around these loads: behind one the compiler has to wait for everything in flight before it may use any of it.
    // Past the last step they repeat it.
    auto fetch = [&](int t, v4i (&a)[LA], v4i (&b)[LB]) {
        const int k = ((t < whole ? t : whole - 1) * KG + kg) * KSTEP + ld_chunk * 16;
#pragma unroll
        for (int i = 0; i < LA; i++) a[i] = load16(pa[i] + k);
#pragma unroll
        for (int i = 0; i < LB; i++) b[i] = load16(pb[i] + k);
    };
    auto put = [&](int t, const v4i (&a)[LA], const v4i (&b)[LB]) {
        int8_t* s = smem + (t & 1) * STEP_BYTES;
#pragma unroll
        for (int i = 0; i < LA; i++) *reinterpret_cast<v4i*>(s + wr_a[i]) = a[i];
#pragma unroll
        for (int i = 0; i < LB; i++) *reinterpret_cast<v4i*>(s + wr_b[i]) = b[i];
    };

    // a wavefront with a single block keeps two sums of it: a product need not wait for the one before
    constexpr int SETS = TM * TN == 1 ? 2 : 1;
    v16i accs[SETS][TM][TN];
    v16i(&acc)[TM][TN] = accs[0];
#pragma unroll
    for (int s = 0; s < SETS; s++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) accs[s][i][j][r] = 0;
    int rd[4];
#pragma unroll
    for (int q = 0; q < 4; q++) rd[q] = l32 * KSTEP + (((2 * q + lhi) ^ (l32 >> 1)) & 7) * 16;
    auto multiply = [&](int t) {
        const int8_t* sa = smem + (t & 1) * STEP_BYTES + wm * (BM / 2) * KSTEP;
        const int8_t* sb = smem + (t & 1) * STEP_BYTES + (BM + wn * (BN / 2)) * KSTEP;
#pragma unroll
        for (int q = 0; q < 4; q++)
        {
            v4i fa[TM], fb[TN];
#pragma unroll
            for (int i = 0; i < TM; i++) fa[i] = *reinterpret_cast<const v4i*>(sa + i * 32 * KSTEP + rd[q]);
#pragma unroll
            for (int j = 0; j < TN; j++) fb[j] = *reinterpret_cast<const v4i*>(sb + j * 32 * KSTEP + rd[q]);
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) accs[q % SETS][i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[i], fb[j], accs[q % SETS][i][j], 0, 0, 0);
        }
    };

    if (whole)
    {
#pragma unroll
        for (int s = 0; s < AHEAD; s++) fetch(s, ra[s], rb[s]);
        put(0, ra[0], rb[0]);
    }
    __syncthreads();
    for (int t0 = 0; t0 < turns; t0 += AHEAD)
    {
#pragma unroll
        for (int u = 0; u < AHEAD; u++)
        {
            const int t = t0 + u; // its registers, ra[u], went to LDS in the turn before
            if (t >= turns) break;
            fetch(t + AHEAD, ra[u], rb[u]);
            if (KG == 1 || t < whole) multiply(t);
            if (t + 1 < whole) put(t + 1, ra[(u + 1) % AHEAD], rb[(u + 1) % AHEAD]);
            __syncthreads();
        }
    }
    if (K != whole_all * KSTEP)
    {
        const int drop = tail_drop < 0 ? 0 : tail_drop > 16 ? 16 : tail_drop;
#pragma unroll
        for (int i = 0; i < LA; i++) ta[i] = drop_bytes(ta[i], drop);
#pragma unroll
        for (int i = 0; i < LB; i++) tb[i] = drop_bytes(tb[i], drop);
        if (tail) put(whole, ta, tb);
        __syncthreads();
        if (tail) multiply(whole);
    }

    if (SETS == 2)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[0][0][r] += accs[SETS - 1][0][0][r];

    if (KG > 1)
    {
        __syncthreads(); // the buffers are free
        int* sums = reinterpret_cast<int*>(smem);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < 16; r++)
                    sums[(wm * (BM / 2) + i * 32 + 8 * (r >> 2) + 4 * lhi + (r & 3)) * BN + wn * (BN / 2) + j * 32 + l32] = acc[i][j][r];
        __syncthreads();
        // every thread finishes one column of the tile, every (256 * KG / BN)-th row
        const int in_col = threadIdx.x % BN, col = col0 + in_col;
        if (col >= N) return;
        float scale, add;
        epi.column(col, scale, add);
        const int* all = reinterpret_cast<const int*>(smem_all) + in_col;
#pragma unroll 4
        for (int in_tile = threadIdx.x / BN; in_tile < BM; in_tile += 256 * KG / BN)
        {
            if (row0 + in_tile >= M) break;
            int v = 0;
#pragma unroll
            for (int g = 0; g < KG; g++) v += all[g * (2 * STEP_BYTES / 4) + in_tile * BN];
            epi.store(row0 + in_tile, col, v, row_value[in_tile], scale, add);
        }
        return;
    }

#pragma unroll
    for (int j = 0; j < TN; j++)
    {
        const int col = col0 + wn * (BN / 2) + j * 32 + l32;
        float scale = 0.f, add = 0.f;
        if (col < N) epi.column(col, scale, add);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int r = 0; r < 16; r++)
            {
                const int in_tile = wm * (BM / 2) + i * 32 + 8 * (r >> 2) + 4 * lhi + (r & 3);
                if (row0 + in_tile < M && col < N) epi.store(row0 + in_tile, col, acc[i][j][r], row_value[in_tile], scale, add);
            }
    }
}

// K below 16: a thread per output
template<typename Epilogue>
__global__ __launch_bounds__(256) void gemm_int8_short_k_kernel(const int8_t* __restrict__ A, size_t lda, const int8_t* __restrict__ B, size_t ldb, int M, int N, int K,
                                                                Epilogue epi)
{
    const size_t o = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (o >= (size_t)M * N) return;
    const int i = (int)(o / N), j = (int)(o % N);
    int acc = 0;
    for (int k = 0; k < K; k++) acc += (int)A[(size_t)i * lda + k] * (int)B[(size_t)j * ldb + k];
    float scale, add;
    epi.column(j, scale, add);
    epi.store(i, j, acc, epi.row_value(i), scale, add);
}

template<int BM, int BN, int KG, typename Epilogue>
static int launch_tile(const int8_t* a, size_t lda, const int8_t* b, size_t ldb, int M, int N, int K, const Epilogue& epi, hipStream_t stream)
{
    const long long tm = ceil_div(M, BM), tn = ceil_div(N, BN);
    NCNNHIP_REQUIRE(tm * tn <= 0x7fffffff, "int8 Gemm: %d x %d outputs are too many tiles", M, N);
    hipLaunchKernelGGL((gemm_int8_general_kernel<BM, BN, KG, Epilogue>), dim3((unsigned)(tm * tn)), dim3(256 * KG), 0, stream, a, lda, b, ldb, M, N, K, (int)tm, (int)tn, epi);
    return launch_status("gemm_int8_general_kernel");
}

template<typename Epilogue>
static int launch_any(const int8_t* a, size_t lda, const int8_t* b, size_t ldb, int M, int N, int K, const Epilogue& epi, hipStream_t stream)
{
    if (K < 16)
    {
        const size_t blocks = ((size_t)M * N + 255) / 256;
        NCNNHIP_REQUIRE(blocks <= 0x7fffffff, "int8 Gemm: %d x %d outputs", M, N);
        hipLaunchKernelGGL((gemm_int8_short_k_kernel<Epilogue>), dim3((unsigned)blocks), dim3(256), 0, stream, a, lda, b, ldb, M, N, K, epi);
        return launch_status("gemm_int8_short_k_kernel");
    }
    // 64 x 64 tiles keep the most compute units busy and are the fastest up to about six of them per unit; beyond that the
    // operand bytes per product decide, half as many with 128 x 128 tiles (2000 x 4000 x 4096: 74 -> 53 us, 2500 cubed 56 ->
    // 41, 2048 cubed the same 20).  With few tiles and a long K two groups of wavefronts halve the chain of steps (96 x 8192
    // x 8192 26 -> 21.5, 1100 x 520 x 7000 23.4 -> 20.2; 333 x 777 x 999 7.4 -> 8.6: not below some 24 steps).
    const long long tiles = (long long)ceil_div(M, 64) * ceil_div(N, 64);
    if (tiles >= 1536) return launch_tile<128, 128, 1>(a, lda, b, ldb, M, N, K, epi, stream);
    if (tiles <= 512 && K >= 3072) return launch_tile<64, 64, 2>(a, lda, b, ldb, M, N, K, epi, stream);
    return launch_tile<64, 64, 1>(a, lda, b, ldb, M, N, K, epi, stream);
}

int launch_gemm_int8_general(const int8_t* a, size_t lda, const int8_t* b, size_t ldb, int M, int N, int K, const GemmEpilogue& epi, hipStream_t stream)
{
    if (!epi.transpose && !epi.acc_out && (epi.bt == -1 || epi.bt == 0 || epi.bt == 4))
        return launch_any(a, lda, b, ldb, M, N, K, TileGemm<true>{epi}, stream);
    return launch_any(a, lda, b, ldb, M, N, K, TileGemm<false>{epi}, stream);
}

int launch_fc_int8_general(const int8_t* x, size_t xs, const int8_t* w, size_t ws, int rows, int num_output, int K, const FcEpilogue& epi, hipStream_t stream)
{
    return launch_any(x, xs, w, ws, rows, num_output, K, TileFc{epi}, stream);
}

} // namespace ncnnhip
