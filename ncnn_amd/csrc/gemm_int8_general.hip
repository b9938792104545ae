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
// Bound by latency and by the first-level cache at the sizes it is for (some hundred tiles of 64 x 64; two workgroups on one unit bring it
// 720 cycles of lines a step, and a step takes 960): 1501 x 1000 x 2008 168 us with the byte gathers of the kernel before this one, 13.1
// -> 12.5 since two products' operands are read at once and the rows' values in one go.  Fewer tiles go to gemm_int8_stream_kernel below.
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
    // a wavefront's share is BM / 2 x BN / 2, in blocks of 32 x 32 or, where that does not divide it, 16 x 16 (as many cycles and operand bytes a product)
    constexpr int BLK = BM % 64 == 0 && BN % 64 == 0 ? 32 : 16;
    constexpr int TM = BM / 2 / BLK, TN = BN / 2 / BLK;
    constexpr int REGS = BLK * BLK / 64;
    typedef int block_sums __attribute__((ext_vector_type(REGS)));
    constexpr int LA = BM / 32, LB = BN / 32;     // 16-byte loads per thread and operand: 32 rows of 8 chunks at a time
    constexpr int STEP_BYTES = (BM + BN) * KSTEP;
    static_assert(KG == 1 || BM * BN * 4 <= 2 * STEP_BYTES, "the sums of a group fit its buffers");
    __shared__ __attribute__((aligned(16))) int8_t smem_all[KG * 2 * STEP_BYTES];
    __shared__ __attribute__((aligned(16))) float row_value[BM];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3);
    const int kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    int8_t* smem = smem_all + kg * 2 * STEP_BYTES;
    const int wm = wave >> 1, wn = wave & 1, lrow = lane & (BLK - 1), lhi = lane / BLK; // lhi: K chunk of the lane, and its rows of the sums

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
    block_sums accs[SETS][TM][TN];
    block_sums(&acc)[TM][TN] = accs[0];
#pragma unroll
    for (int s = 0; s < SETS; s++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < REGS; r++) accs[s][i][j][r] = 0;
    constexpr int PARTS = BLK == 32 ? 4 : 2, CHUNKS = 8 / PARTS; // parts of a K step that one product takes, and their chunks
    int rd[PARTS];
#pragma unroll
    for (int q = 0; q < PARTS; q++) rd[q] = lrow * KSTEP + (((CHUNKS * q + lhi) ^ (lrow >> 1)) & 7) * 16;
    auto multiply = [&](int t) {
        const int8_t* sa = smem + (t & 1) * STEP_BYTES + wm * (BM / 2) * KSTEP;
        const int8_t* sb = smem + (t & 1) * STEP_BYTES + (BM + wn * (BN / 2)) * KSTEP;
        // Q parts of the step are read before they are multiplied: left to itself the compiler reads two operands, waits, multiplies and
        // reads the next two into the same registers.  As many as leave the workgroups a unit holds their registers.
        constexpr int Q = (TM * TN == 1 && KG == 1) || BLK == 16 ? 2 : 1;
#pragma unroll
        for (int q0 = 0; q0 < PARTS; q0 += Q)
        {
            v4i fa[Q][TM], fb[Q][TN];
#pragma unroll
            for (int q = 0; q < Q; q++)
            {
#pragma unroll
                for (int i = 0; i < TM; i++) fa[q][i] = *reinterpret_cast<const v4i*>(sa + i * BLK * KSTEP + rd[q0 + q]);
#pragma unroll
                for (int j = 0; j < TN; j++) fb[q][j] = *reinterpret_cast<const v4i*>(sb + j * BLK * KSTEP + rd[q0 + q]);
            }
            if (Q > 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < Q; q++)
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
                    {
                        block_sums& sum = accs[(q0 + q) % SETS][i][j];
                        if constexpr (BLK == 32)
                            sum = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[q][i], fb[q][j], sum, 0, 0, 0);
                        else
                            sum = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[q][i], fb[q][j], sum, 0, 0, 0);
                    }
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
        for (int r = 0; r < REGS; r++) acc[0][0][r] += accs[SETS - 1][0][0][r];

    if (KG > 1)
    {
        __syncthreads(); // the buffers are free
        int* sums = reinterpret_cast<int*>(smem);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < REGS; r++)
                    sums[(wm * (BM / 2) + i * BLK + 8 * (r >> 2) + 4 * lhi + (r & 3)) * BN + wn * (BN / 2) + j * BLK + lrow] = acc[i][j][r];
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

    // the rows' values in one go, four consecutive ones at a time
    typedef float v4f_rows __attribute__((ext_vector_type(4)));
    v4f_rows rows[TM][REGS / 4];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int e = 0; e < REGS / 4; e++) rows[i][e] = *reinterpret_cast<const v4f_rows*>(row_value + wm * (BM / 2) + i * BLK + 8 * e + 4 * lhi);
#pragma unroll
    for (int j = 0; j < TN; j++)
    {
        const int col = col0 + wn * (BN / 2) + j * BLK + lrow;
        if (col >= N) continue;
        float scale, add;
        epi.column(col, scale, add);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int r = 0; r < REGS; r++)
            {
                const int in_tile = wm * (BM / 2) + i * BLK + 8 * (r >> 2) + 4 * lhi + (r & 3);
                if (row0 + in_tile < M) epi.store(row0 + in_tile, col, acc[i][j][r], rows[i][r >> 2][r & 3], scale, add);
            }
    }
}

// Between a wavefront's writes to its own piece of LDS and its reads of what other lanes wrote there: LDS serves a wavefront in order, so no
// instruction comes of it, but the compiler may not move memory accesses across it either.
__device__ __forceinline__ void exchange_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Few tiles (gemm_int8_streams): the W wavefronts of a workgroup each multiply the whole BM x BN tile over a run of K steps of their own.
// A wavefront fetches 128 bytes of each of its rows into registers (coalesced, any alignment), turns them into the operand mapping through
// a piece of LDS that belongs to it alone -- LDS serves a wavefront in order, so no barrier stands in the loop -- and requests the next
// step before it multiplies.  The sums meet in LDS at the end.  Bound by latency: a launch, one trip to memory for every one to four
// steps, the sums; 32 x 32 tiles put four times as many workgroups on the chip as 64 x 64.
template<int BM, int BN, int W, typename Epilogue>
__global__ __launch_bounds__(64 * W) void gemm_int8_stream_kernel(const int8_t* __restrict__ A, size_t lda, const int8_t* __restrict__ B, size_t ldb, int M, int N, int K,
                                                                  Epilogue epi)
{
    constexpr int TM = BM / 32, TN = BN / 32; // 32 x 32 blocks
    constexpr int LA = BM / 8, LB = BN / 8;   // loads of 8 rows x 128 bytes
    constexpr int STEP_BYTES = (BM + BN) * KSTEP;
    static_assert(BM * BN * 4 <= STEP_BYTES, "a wavefront's sums fit its piece of LDS");
    __shared__ __attribute__((aligned(16))) int8_t smem_all[W * STEP_BYTES];
    __shared__ float row_value[BM];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, lhi = lane >> 5;
    int8_t* smem = smem_all + wave * STEP_BYTES;

    const int row0 = blockIdx.y * BM, col0 = blockIdx.x * BN;

    // this wavefront's K steps; the last of all may end inside: its chunks beyond K are fetched from the row's end and cut when they go to LDS
    const int all = (K + KSTEP - 1) / KSTEP;
    const int step0 = all * wave / W, steps = all * (wave + 1) / W - step0;
    const int cut_step = K % KSTEP ? all - 1 - step0 : -1;
    const int ld_row = lane >> 3, ld_chunk = lane & 7;
    const int8_t* pa = A + (size_t)row0 * lda;
    const int8_t* pb = B + (size_t)col0 * ldb;
    size_t off_a[LA], off_b[LB];
#pragma unroll
    for (int i = 0; i < LA; i++) off_a[i] = (size_t)(row0 + i * 8 + ld_row < M ? i * 8 + ld_row : M - 1 - row0) * lda;
#pragma unroll
    for (int i = 0; i < LB; i++) off_b[i] = (size_t)(col0 + i * 8 + ld_row < N ? i * 8 + ld_row : N - 1 - col0) * ldb;
    v4i ra[LA], rb[LB];
    auto fetch = [&](int t) {
        const int k = (step0 + (t < steps ? t : 0)) * KSTEP + ld_chunk * 16;
        const int kk = k < K - 16 ? k : K - 16;
#pragma unroll
        for (int i = 0; i < LA; i++) ra[i] = load16(pa + off_a[i] + kk);
#pragma unroll
        for (int i = 0; i < LB; i++) rb[i] = load16(pb + off_b[i] + kk);
    };
    fetch(0);

    // what the end needs besides the sums
    const int in_col = threadIdx.x % BN, col = col0 + in_col;
    if ((int)threadIdx.x < BM) row_value[threadIdx.x] = row0 + (int)threadIdx.x < M ? epi.row_value(row0 + threadIdx.x) : 0.f;
    float scale = 0.f, add = 0.f;
    if (col < N) epi.column(col, scale, add);

    v16i acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0;
    // row r of an operand keeps chunk c at position c ^ ((r >> 1) & 7): r = i * 8 + ld_row when written, i * 32 + l32 when read
    const int wr0 = ld_row * KSTEP + (ld_chunk ^ (ld_row >> 1)) * 16, wr1 = ld_row * KSTEP + (ld_chunk ^ (ld_row >> 1) ^ 4) * 16;
    int rd[4];
#pragma unroll
    for (int q = 0; q < 4; q++) rd[q] = l32 * KSTEP + (((2 * q + lhi) ^ (l32 >> 1)) & 7) * 16;

    for (int t = 0; t < steps; t++)
    {
        if (t == cut_step) // uniform
        {
            const int over = (step0 + t) * KSTEP + ld_chunk * 16 + 16 - K, drop = over < 0 ? 0 : over > 16 ? 16 : over;
#pragma unroll
            for (int i = 0; i < LA; i++) ra[i] = drop_bytes(ra[i], drop);
#pragma unroll
            for (int i = 0; i < LB; i++) rb[i] = drop_bytes(rb[i], drop);
        }
#pragma unroll
        for (int i = 0; i < LA; i++) *reinterpret_cast<v4i*>(smem + i * 1024 + (i & 1 ? wr1 : wr0)) = ra[i];
#pragma unroll
        for (int i = 0; i < LB; i++) *reinterpret_cast<v4i*>(smem + BM * KSTEP + i * 1024 + (i & 1 ? wr1 : wr0)) = rb[i];
        exchange_fence();
        fetch(t + 1); // (past the last step: the first again)
        v4i fa[4][TM], fb[4][TN]; // every read before the first product, as above
#pragma unroll
        for (int q = 0; q < 4; q++)
        {
#pragma unroll
            for (int i = 0; i < TM; i++) fa[q][i] = *reinterpret_cast<const v4i*>(smem + i * 32 * KSTEP + rd[q]);
#pragma unroll
            for (int j = 0; j < TN; j++) fb[q][j] = *reinterpret_cast<const v4i*>(smem + (BM + j * 32) * KSTEP + rd[q]);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[q][i], fb[q][j], acc[i][j], 0, 0, 0);
        exchange_fence();
    }

    int* sums = reinterpret_cast<int*>(smem);
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) sums[(i * 32 + 8 * (r >> 2) + 4 * lhi + (r & 3)) * BN + j * 32 + l32] = acc[i][j][r];
    __syncthreads();
    if (col >= N) return;
    // every thread finishes one column of the tile, every (64 * W / BN)-th row
    const int* from = reinterpret_cast<const int*>(smem_all) + in_col;
#pragma unroll 4
    for (int in_tile = threadIdx.x / BN; in_tile < BM; in_tile += 64 * W / BN)
    {
        if (row0 + in_tile >= M) break;
        int v = 0;
#pragma unroll
        for (int w = 0; w < W; w++) v += from[w * (STEP_BYTES / 4) + in_tile * BN];
        epi.store(row0 + in_tile, col, v, row_value[in_tile], scale, add);
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

template<int BM, int BN, int W, typename Epilogue>
static int launch_stream(const int8_t* a, size_t lda, const int8_t* b, size_t ldb, int M, int N, int K, const Epilogue& epi, hipStream_t stream)
{
    const long long tm = ceil_div(M, BM), tn = ceil_div(N, BN);
    hipLaunchKernelGGL((gemm_int8_stream_kernel<BM, BN, W, Epilogue>), dim3((unsigned)tn, (unsigned)tm), dim3(64 * W), 0, stream, a, lda, b, ldb, M, N, K, epi);
    return launch_status("gemm_int8_stream_kernel");
}

static inline bool rows_aligned16(const int8_t* p, size_t stride, int K)
{
    return (reinterpret_cast<uintptr_t>(p) & 15) == 0 && stride % 16 == 0 && K % 16 == 0;
}

// Where the streaming kernel is the quicker one.  Up to 16 rows always: it reads B once, at 5.5 TB/s where B is large (one or two rows on few
// columns with K beyond 5000 pay for its serial steps: 1 x 1656 x 8000 7.1 us, 6.1 with 16 columns a workgroup; sixteen wavefronts a tile instead
// of eight took 1 to 13 % longer).  Else by its tiles: it
// reads the operands of each 32 x 32 tile, four times the bytes a product that 128 x 128 tiles read, and rows off 16 bytes cost two cache
// lines for one.  us, Gemm alone, the quickest other kernel here -> this one: 1 x 8192 x 8192 16.5 -> 12.0, 32 x 4096 x 4096 11.0 -> 5.8, 64 x 512
// x 512 5.2 -> 4.6, 281 x 720 x 2048 8.8 -> 4.6, 360 x 936 x 4672 13.9 -> 10.1, 551 x 1024 x 2048 9.0 -> 7.6, 1024 cubed 8.2 -> 6.8, 512 x
// 2048 x 2048 11.1 -> 8.9; 256 x 4096 x 4096 17.3 -> 12.2 with 64 x 64 tiles and eight wavefronts; off 16 bytes 16 x 8000 x 8001 42 -> 17, 895 x
// 456 x 473 6.5 -> 5.8; and where it is not taken: 1226 x 1344 x 2944 17.0 -> 18.0, 330 x 6616 x 896 10.2 -> 11.7, 2284 x 336 x 1216 7.4 ->
// 7.9, off 16 bytes 148 x 3311 x 537 6.8 -> 7.8.  With a long K it is left from two cut tiles a unit on (22 shapes of 515 to 638 tiles, K 2944 to 7808: 5 %
// less here in one, 3 to 35 % more in the others: 192 x 2960 x 4480 13.0 -> 17.6, 131 x 3848 x 6464 18.4 -> 24.1, 1369 x 440 x 3392 11.3 -> 13.4; at
// 480 to 510 tiles from 26 % less to 14 % more; of whole multiples of 128 up to 14 % less, 5 % more at worst: 256 x 2304 x 6144 16.5 ->
// 14.5).  (From 640 to 1024 tiles it is better than the 128 x 128 tiles of whole multiples, not than 64 x 64.)  Eight wavefronts a tile
// up to one tile a unit and from nine K steps (128 x 1024 x 4096 5.7, four 6.2), else four.
bool gemm_int8_streams(int M, int N, int K, bool aligned)
{
    if (K < 16) return false;
    if (M <= 16) return true;
    const long long tiles32 = (long long)ceil_div(M, 32) * ceil_div(N, 32);
    if (!aligned) return tiles32 <= 450;
    if (M % 128 == 0 && N % 128 == 0) return tiles32 <= 1024;
    return tiles32 <= (K >= 2944 ? 512 : 640);
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
    const bool aligned = rows_aligned16(a, lda, K) && rows_aligned16(b, ldb, K);
    if (gemm_int8_streams(M, N, K, aligned))
    {
        const long long tiles32 = (long long)ceil_div(M, 32) * ceil_div(N, 32);
        if (M > 16 && tiles32 > 640 && K >= 3072) return launch_stream<64, 64, 8>(a, lda, b, ldb, M, N, K, epi, stream);
        if (tiles32 <= 256 && K > 1024) return launch_stream<32, 32, 8>(a, lda, b, ldb, M, N, K, epi, stream);
        return launch_stream<32, 32, 4>(a, lda, b, ldb, M, N, K, epi, stream);
    }
    // 64 x 64 tiles keep the most compute units busy and are the fastest up to about six of them per unit; beyond that the
    // operand bytes per product decide, half as many with 128 x 128 tiles (2000 x 4000 x 4096: 74 -> 53 us, 2500 cubed 56 ->
    // 41, 2048 cubed the same 20).  With few tiles and a long K two groups of wavefronts halve the chain of steps (1100 x 520 x 7000
    // 23.4 -> 20.2; not below some 24 steps).
    // Rows off 16 bytes cost up to 2 times the cache lines, rows off 4 bytes 2.4 times the cycles of aligned ones (834 against 346 for 16 KB), and
    // the bytes decide earlier: while one round of 128 x 128 tiles does it, from 800 tiles (2048 x 2048 x 2004 23.9 -> 20.1, 1792 x 2048 x 1004
    // 14.3 -> 13.6; 768 tiles 19.2 18.4, 640 x 1004 11.9 12.8), off 4 bytes from 600 (1280 x 2048 x 2003 25.1 -> 22.5, 2048 x 2048 x 3001 42.6 ->
    // 32.1), with more rounds from 1300 (2816 x 2048 x 2004 32.0 -> 28.2; 1152 tiles the same), and not on a short K (2048 x 2048 x 508 10.7 11.8).
    const long long tiles = (long long)ceil_div(M, 64) * ceil_div(N, 64), tiles128 = (long long)ceil_div(M, 128) * ceil_div(N, 128);
    const bool words = ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) | lda | ldb) & 3) == 0;
    // Tiles between the two where 64 x 64 ones would be two to some units and these are one to each: with 96 x 64 a unit reads 160 rows a step for 256.  us, 64 x 64 -> 96 x 64: off
    // 16 bytes 1501 x 1000 x 2008 12.7 -> 11.7, 299 x 3801 x 389 8.7 -> 7.8, 2362 x 540 x 271 8.2 -> 7.4; aligned, two groups of wavefronts on a long K, 855 x 1504 x 6464
    // 28.3 -> 22.3, 811 x 1544 x 6208 27.6 -> 21.5, 1294 x 1136 x 960 8.5 -> 8.3, and not on a short K, 999 x 1312 x 512 6.3 -> 6.6.  Off 16 bytes 96 x 96 for three and
    // more 64 x 64 to a unit: 2902 x 740 x 1254 16.2 -> 12.8, 539 x 3870 x 549 12.9 -> 10.9, 264 x 7947 x 427 11.8 -> 10.1 (aligned 795 x 2608 x 704 9.3 -> 9.9).
    const long long tiles96 = (long long)ceil_div(M, 96) * ceil_div(N, 64);
    if (tiles > 256 && tiles <= 512 && tiles96 <= 256 && (aligned ? K >= 900 : K > 256))
    {
        if (K >= 3072) return launch_tile<96, 64, 2>(a, lda, b, ldb, M, N, K, epi, stream);
        return launch_tile<96, 64, 1>(a, lda, b, ldb, M, N, K, epi, stream);
    }
    if (!aligned && tiles > 512 && K >= 400 && (long long)ceil_div(M, 96) * ceil_div(N, 96) <= 256) return launch_tile<96, 96, 1>(a, lda, b, ldb, M, N, K, epi, stream);
    if (!aligned && K >= 1000 && tiles >= (tiles128 > 256 ? 1300 : words ? 800 : 600)) return launch_tile<128, 128, 1>(a, lda, b, ldb, M, N, K, epi, stream);
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
