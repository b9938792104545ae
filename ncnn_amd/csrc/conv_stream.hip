// int8 Convolution (group 1, zero border) on channels-last blobs, for layers with few output tiles: a workgroup owns 16 or 32 pixels x 16
// or 32 channels and each of its wavefronts multiplies the whole tile over a run of K steps of its own, operands straight from
// global memory into registers in the order the matrix cores take them.
//
// Bound by latency: with no more tiles than compute units nothing overlaps a tile but its own loads, and the pipelined kernel
// (conv_nhwc_pipelined_kernel.h) walks K behind a barrier per 64 bytes, about 190 ns each, where here a layer is one trip to memory, a few
// dozen matrix instructions, one meeting of the sums in LDS and the epilogue.
//
// v_mfma_i32_16x16x64_i8 with weights as the A operand: a lane's four results are four neighbouring channels of one pixel, so the
// epilogue needs no transpose: four entries of each table, one 16-byte fp32 store and residual load, one 4-byte int8 store.
//
// One trip to memory means one: every load of the tile, the epilogue's tables among them, is issued before the first product (left alone the compiler
// puts products between the loads and waits for each, which was a second trip).  Loads go through buffer descriptors: a step is an immediate offset, and what lies
// outside the image, the run of steps or the tables is an offset beyond the buffer, which answers zero without a fetch.  us in a captured chain, weights from HBM,
// before / here: 1x1 512 -> 128 on 28 x 28 3.7 / 2.9, 1024 -> 256 on 14 x 14 3.7 / 2.9, 256 -> 1024 with the fused tail 4.1 / 3.0, 3x3 256 -> 256 4.6 / 4.0,
// 3x3 512 -> 512 on 7 x 7 7.2 / 6.4, 1x1 512 -> 2048 4.4 / 3.2, 960 -> 160 3.2 / 2.4; inside a workgroup the operands arrive 1.9 to 3.1 us after its first
// instruction before and 1.2 to 2 here, of which 0.25 were the arguments and 1.4 the issue of loads between waits.
#include "conv_nhwc.h"

namespace ncnnhip {

typedef int v4i_cs __attribute__((ext_vector_type(4)));
typedef float v4f_cs __attribute__((ext_vector_type(4)));

constexpr unsigned BEYOND = 0x80000000u; // an offset beyond every buffer here (their sizes are below 2^31: stream_reaches)

static __device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, unsigned bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
static __device__ __forceinline__ v4i_cs load16(__amdgpu_buffer_rsrc_t buffer, unsigned offset)
{
    return __builtin_bit_cast(v4i_cs, __builtin_amdgcn_raw_buffer_load_b128(buffer, (int)offset, 0, 0));
}
static __device__ __forceinline__ float load_float(__amdgpu_buffer_rsrc_t buffer, unsigned offset)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(buffer, (int)offset, 0, 0));
}

// How a step of 64 bytes of K finds its pixels where the layer is not dense.
struct StreamTaps
{
    int H, W, kw, dh, dw, sh, sw, pad_top, pad_left, outw, plane; // plane: output pixels of an image
    int steps; // of one tap
    unsigned magic_plane, magic_outw, magic_steps, magic_kw;
};

// n / d for n below 2^16 or so, d == 1 ? n : n * (2^32 / d + 1) >> 32, exact while n * d < 2^32
static __device__ __forceinline__ int magic_div(int n, int d, unsigned magic)
{
    return d == 1 ? n : (int)__umulhi((unsigned)n, magic);
}
static unsigned magic_of(int d)
{
    return d > 1 ? (unsigned)((1ull << 32) / (unsigned)d + 1) : 0u;
}

// A shortcut as the kernel walks it.
struct StreamShortcut : ConvShortcut
{
    unsigned x_bytes;
    int per_wave; // steps
    int plane;
    unsigned magic_plane, magic_outw;
};
template<bool PRESENT>
struct StreamShortcutArg
{
};
template<>
struct StreamShortcutArg<true> : StreamShortcut
{
};

// What a workgroup needs once its operands are on their way, and how it finds them where that is not simple.
struct StreamEpilogue
{
    const float* scale_in;
    const float* bias;
    const float* scale_out;
    const float* residual;
    void* out;
    int8_t* q8_out;
    float q8_scale;
    int relu_after;
    ncnnhip_activation act;
};
template<bool SHORTCUT>
struct StreamRest
{
    StreamEpilogue epi;
    StreamShortcutArg<SHORTCUT> shortcut;
    StreamTaps taps;
};

// DENSE: 1x1, stride 1, unpadded: output pixel = input pixel.  Otherwise taps of whole 64-byte steps, so that a step lies inside one tap.
// TP, TC: 16-pixel and 16-channel blocks of a tile.  U: K steps a wavefront has in flight, at 4 (TP + TC) registers each; W: wavefronts.
// SHORTCUT: a projection shortcut is added (ConvShortcut), its K dealt out to the wavefronts and its sums met in the same way; both convolutions'
// loads are in flight together.
// The arguments before `rest` are REST_AT bytes and arrive in registers (amdgpu-kernarg-preload-count), so that the first loads wait for no other; of
// `rest` the epilogue's part is read behind them, through a pointer that the compiler cannot move the reads across.
constexpr size_t REST_AT = 56;
template<bool DENSE, int TP, int TC, int U, int W, bool SHORTCUT = false>
__global__ __launch_bounds__(64 * W) void conv_stream_kernel(const int8_t* __restrict__ wpk, const int8_t* __restrict__ x, unsigned x_bytes, int K, int Cp, int npix, int cout,
                                                             int out_cp, int tiles, int tiles_m, unsigned magic_m, int per_wave,
                                                             StreamRest<SHORTCUT> rest)
{
    constexpr int NB = TP * TC; // 16 x 16 blocks of the tile
    static_assert(NB <= W, "a wavefront finishes one block");
    static_assert(!SHORTCUT || DENSE, "the sum's main convolution is 1x1");
    __shared__ v4i_cs part[SHORTCUT ? 2 : 1][W][NB][64]; // [wavefront][block][lane]
    const int lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // XCD x gets the x-th contiguous share of the tiles, the pixel tiles of one channel tile side by side: its weights cross to one XCD
    int b = blockIdx.x;
    {
        const int xcd = b & 7, idx = b >> 3, rem = tiles & 7;
        b = xcd * (tiles >> 3) + (xcd < rem ? xcd : rem) + idx;
    }
    const int tn = magic_div(b, tiles_m, magic_m);
    const int pix0 = (b - tn * tiles_m) * (16 * TP), ch0 = tn * (16 * TC);

    const int total = K / 64;
    int s0 = wave * per_wave;
    const int end = s0 + per_wave < total ? s0 + per_wave : total;

    const __amdgpu_buffer_rsrc_t w_buf = buffer_of(wpk, (unsigned)(cout * K)), x_buf = buffer_of(x, x_bytes);
    const StreamTaps& g = rest.taps;
    unsigned beyond = BEYOND;
    asm volatile("" : "+v"(beyond)); // (in a register: steps stay immediate offsets)
    unsigned w_off[TC], x_off[TP]; // dense: the pixel's bytes of step s0; else those of its first tap's channels
    int iy0[TP], ix0[TP];
#pragma unroll
    for (int i = 0; i < TC; i++)
    {
        const int ch = ch0 + i * 16 + r16;
        w_off[i] = ch < cout ? (unsigned)(ch * K + s0 * 64 + kq * 16) : beyond;
    }
#pragma unroll
    for (int i = 0; i < TP; i++)
    {
        const int p = pix0 + i * 16 + r16;
        if (DENSE)
            x_off[i] = p < npix ? (unsigned)(p * Cp + s0 * 64 + kq * 16) : beyond; // (the last step may reach into the next pixel, whose bytes meet zero weights)
        else
        {
            const int img = magic_div(p, g.plane, g.magic_plane), at = p - img * g.plane, oy = magic_div(at, g.outw, g.magic_outw);
            iy0[i] = p < npix ? oy * g.sh - g.pad_top : -0x40000000; // a pixel beyond the last fails every bounds test
            ix0[i] = (at - oy * g.outw) * g.sw - g.pad_left;
            x_off[i] = ((unsigned)(img * g.H + iy0[i]) * (unsigned)g.W + (unsigned)ix0[i]) * (unsigned)Cp + kq * 16; // (modulo 2^32: a tap's offset brings it back into the image)
        }
    }
    int q = 0, ky = 0, kx = 0; // step inside the tap, and the tap: the same in every lane
    if (!DENSE)
    {
        const int tap = magic_div(s0, g.steps, g.magic_steps);
        q = s0 - tap * g.steps;
        ky = magic_div(tap, g.kw, g.magic_kw);
        kx = tap - ky * g.kw;
    }

    v4i_cs fw[U][TC], fx[U][TP];
    auto issue = [&] {
#pragma unroll
        for (int u = 0; u < U; u++)
        {
            const bool live = s0 + u < end; // a step beyond the run is nothing but zeros
#pragma unroll
            for (int i = 0; i < TC; i++) fw[u][i] = load16(w_buf, (live ? w_off[i] : beyond) + u * 64);
            if (DENSE)
            {
#pragma unroll
                for (int i = 0; i < TP; i++) fx[u][i] = load16(x_buf, (live ? x_off[i] : beyond) + u * 64);
            }
            else
            {
                const int dy = ky * g.dh, dx = kx * g.dw;
                const unsigned at = (unsigned)((dy * g.W + dx) * Cp + q * 64);
#pragma unroll
                for (int i = 0; i < TP; i++)
                {
                    const bool in = live && (unsigned)(iy0[i] + dy) < (unsigned)g.H && (unsigned)(ix0[i] + dx) < (unsigned)g.W;
                    fx[u][i] = load16(x_buf, in ? x_off[i] + at : beyond);
                }
                if (++q == g.steps)
                {
                    q = 0;
                    if (++kx == g.kw)
                    {
                        kx = 0;
                        ky++;
                    }
                }
            }
        }
        s0 += U;
#pragma unroll
        for (int i = 0; i < TC; i++) w_off[i] += U * 64;
        if (DENSE)
        {
#pragma unroll
            for (int i = 0; i < TP; i++) x_off[i] += U * 64;
        }
    };
    issue();

    __builtin_amdgcn_sched_barrier(0);
    const __attribute__((address_space(4))) char* rest_at = (const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr() + REST_AT;
    asm volatile("" : "+s"(rest_at));
    const StreamRest<SHORTCUT>& late = *(const StreamRest<SHORTCUT>*)rest_at;
    const StreamShortcutArg<SHORTCUT>& shortcut = late.shortcut;
    const float* const scale_in = late.epi.scale_in;
    const float* const bias_at = late.epi.bias;
    const float* const scale_out = late.epi.scale_out;
    const float* const residual = late.epi.residual;
    void* const out = late.epi.out;
    int8_t* const q8_out = late.epi.q8_out;
    const float q8_scale = late.epi.q8_scale;
    const int relu_after = late.epi.relu_after, act_type = late.epi.act.type;
    asm volatile("" ::"s"(scale_in), "s"(bias_at), "s"(scale_out), "s"(residual), "s"(out), "s"(q8_out), "s"(q8_scale), "s"(relu_after), "s"(act_type)); // one read of them all

    v4i_cs sw[SHORTCUT ? U : 1][TC], sx[SHORTCUT ? U : 1][TP];
    unsigned sw_off[TC], sx_off[TP];
    int t0 = 0, t_end = 0;
    auto issue_shortcut = [&] {
        if constexpr (SHORTCUT)
        {
            const __amdgpu_buffer_rsrc_t sw_buf = buffer_of(shortcut.wpk, (unsigned)(cout * shortcut.Cp)), sx_buf = buffer_of(shortcut.x, shortcut.x_bytes);
#pragma unroll
            for (int u = 0; u < U; u++)
            {
                const bool live = t0 + u < t_end;
#pragma unroll
                for (int i = 0; i < TC; i++) sw[u][i] = load16(sw_buf, (live ? sw_off[i] : beyond) + u * 64);
#pragma unroll
                for (int i = 0; i < TP; i++) sx[u][i] = load16(sx_buf, (live ? sx_off[i] : beyond) + u * 64);
            }
            t0 += U;
#pragma unroll
            for (int i = 0; i < TC; i++) sw_off[i] += U * 64;
#pragma unroll
            for (int i = 0; i < TP; i++) sx_off[i] += U * 64;
        }
    };
    if constexpr (SHORTCUT)
    {
        const int steps = shortcut.Cp / 64;
        t0 = wave * shortcut.per_wave;
        t_end = t0 + shortcut.per_wave < steps ? t0 + shortcut.per_wave : steps;
#pragma unroll
        for (int i = 0; i < TC; i++)
        {
            const int ch = ch0 + i * 16 + r16;
            sw_off[i] = ch < cout ? (unsigned)(ch * shortcut.Cp + t0 * 64 + kq * 16) : beyond;
        }
#pragma unroll
        for (int i = 0; i < TP; i++)
        {
            const int p = pix0 + i * 16 + r16, img = magic_div(p, shortcut.plane, shortcut.magic_plane), at = p - img * shortcut.plane, oy = magic_div(at, shortcut.outw, shortcut.magic_outw), ox = at - oy * shortcut.outw;
            sx_off[i] = p < npix ? (unsigned)(((img * shortcut.H + oy * shortcut.sh) * shortcut.W + ox * shortcut.sw) * shortcut.Cp + t0 * 64 + kq * 16) : beyond;
        }
        issue_shortcut();
    }

    // wavefront n < NB finishes block n: what it needs from memory, behind the operands (the others ask for nothing, without a branch: one would make every
    // wavefront's first product wait for its last load)
    const bool finishes = NB == W || wave < NB;
    const int ch4 = ch0 + wave / TP * 16 + 4 * kq, pix = pix0 + wave % TP * 16 + r16;
    float s_in[4], bias[4], s_out[4];
    float sc_in[4], sc_bias[4];
    const bool to_int8 = scale_out != 0, with_residual = !to_int8 && residual != 0;
    const unsigned table = (unsigned)(cout * 4), table_at = finishes ? (unsigned)ch4 * 4 : beyond;
    const __amdgpu_buffer_rsrc_t in_buf = buffer_of(scale_in, table), bias_buf = buffer_of(bias_at, bias_at ? table : 0), out_buf = buffer_of(scale_out, to_int8 ? table : 0);
#pragma unroll
    for (int e = 0; e < 4; e++)
    {
        s_in[e] = load_float(in_buf, table_at + e * 4);
        bias[e] = load_float(bias_buf, table_at + e * 4);
        s_out[e] = load_float(out_buf, table_at + e * 4);
    }
    if constexpr (SHORTCUT)
    {
        const __amdgpu_buffer_rsrc_t sc_buf = buffer_of(shortcut.scale_in, table), sc_bias_buf = buffer_of(shortcut.bias, shortcut.bias ? table : 0);
#pragma unroll
        for (int e = 0; e < 4; e++)
        {
            sc_in[e] = load_float(sc_buf, table_at + e * 4);
            sc_bias[e] = load_float(sc_bias_buf, table_at + e * 4);
        }
    }
    const __amdgpu_buffer_rsrc_t res_buf = buffer_of(residual, with_residual ? (unsigned)(npix * out_cp) * 4 : 0);
    const v4f_cs res = __builtin_bit_cast(v4f_cs, load16(res_buf, finishes && pix < npix && ch4 < out_cp ? (unsigned)(pix * out_cp + ch4) * 4 : beyond));

    v4i_cs acc[NB], other[NB]; // channel block n / TP, pixel block n % TP
#pragma unroll
    for (int n = 0; n < NB; n++) acc[n] = other[n] = v4i_cs{0, 0, 0, 0};
    auto multiply = [&] {
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int n = 0; n < NB; n++) acc[n] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fw[u][n / TP], fx[u][n % TP], acc[n], 0, 0, 0);
    };
    auto multiply_shortcut = [&] {
        if constexpr (SHORTCUT)
        {
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int n = 0; n < NB; n++) other[n] = __builtin_amdgcn_mfma_i32_16x16x64_i8(sw[u][n / TP], sx[u][n % TP], other[n], 0, 0, 0);
        }
    };
    // the first round outside the loops, where its waits count its loads alone; every load above before the first product
    __builtin_amdgcn_sched_barrier(0);
    multiply();
    multiply_shortcut();
    while (SHORTCUT && s0 < end && t0 < t_end)
    {
        issue();
        issue_shortcut();
        __builtin_amdgcn_sched_barrier(0);
        multiply();
        multiply_shortcut();
    }
    // What is left of the longer K goes on alone: loads of steps that are not there cost a round as much as others.  us, with them / here: 512 channels on 7 x 7, 1 + 383 steps 25.8 /
    // 20.7, 16 + 200 17.9 / 15.8; 2048 channels 1 + 100 15.9 / 13.9, 16 + 128 18.5 / 16.5; 256 on 28 x 28, 64 + 16 13.2 / 12.3.  (Without them in the first round, too, 1 + 383 20.2,
    // but 8 + 16 on 2048 channels 5.0 -> 5.1: a branch there makes the first products wait for the last load.)
    while (s0 < end)
    {
        issue();
        __builtin_amdgcn_sched_barrier(0);
        multiply();
    }
    while (SHORTCUT && t0 < t_end)
    {
        issue_shortcut();
        __builtin_amdgcn_sched_barrier(0);
        multiply_shortcut();
    }

    // the wavefronts' sums meet (integer addition: exact in any order)
#pragma unroll
    for (int n = 0; n < NB; n++)
    {
        part[0][wave][n][lane] = acc[n];
        if constexpr (SHORTCUT) part[1][wave][n][lane] = other[n];
    }
    __syncthreads();
    if (!finishes || ch4 >= out_cp || pix >= npix) return;
    v4i_cs sum = part[0][0][wave][lane];
#pragma unroll
    for (int s = 1; s < W; s++) sum += part[0][s][wave][lane];

    // the pipelined kernel's epilogue, statement by statement
    float f[4];
#pragma unroll
    for (int e = 0; e < 4; e++)
    {
        f[e] = mul_rn((float)sum[e], s_in[e]);
        f[e] = add_rn(f[e], bias_at ? bias[e] : -0.f); // no bias: -0, the one value whose addition changes nothing
    }
    if (act_type == 1)
    {
#pragma unroll
        for (int e = 0; e < 4; e++) f[e] = fmaxf(f[e], 0.f);
    }
    else if (act_type != 0)
    {
#pragma unroll
        for (int e = 0; e < 4; e++) f[e] = apply_activation(f[e], late.epi.act);
    }
    const size_t o = (size_t)pix * out_cp + ch4;
    if (to_int8)
    {
#pragma unroll
        for (int e = 0; e < 4; e++) f[e] = mul_rn(f[e], s_out[e]);
        float2int8_as_float_x4(f[0], f[1], f[2], f[3]);
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (ch4 + e >= cout) f[e] = 0.f; // channels from cout up to out_cp are the blob's zero padding
        *reinterpret_cast<uint32_t*>(static_cast<int8_t*>(out) + o) = pack4_quantised(f[0], f[1], f[2], f[3]);
        return;
    }
    v4f_cs v;
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = ch4 + e < cout ? f[e] : 0.f;
    if constexpr (SHORTCUT)
    {
        v4i_cs sc = part[1][0][wave][lane];
#pragma unroll
        for (int s = 1; s < W; s++) sc += part[1][s][wave][lane];
#pragma unroll
        for (int e = 0; e < 4; e++)
        {
            float t = add_rn(mul_rn((float)sc[e], sc_in[e]), shortcut.bias ? sc_bias[e] : -0.f);
            if (shortcut.act.type != 0) t = apply_activation(t, shortcut.act);
            v[e] = add_rn(v[e], ch4 + e < cout ? t : 0.f);
        }
    }
    if (with_residual)
    {
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = add_rn(v[e], res[e]);
    }
    if (relu_after)
    {
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = v[e] < 0.f ? 0.f : v[e]; // the ReLU LAYER's statement (src/layer/relu.cpp:36-37): a NaN stays, unlike fmaxf
    }
    if (out) *reinterpret_cast<v4f_cs*>(static_cast<float*>(out) + o) = v;
    if (q8_out)
    {
        float q[4];
#pragma unroll
        for (int e = 0; e < 4; e++) q[e] = mul_rn(v[e], q8_scale);
        float2int8_as_float_x4(q[0], q[1], q[2], q[3]);
        *reinterpret_cast<uint32_t*>(q8_out + o) = pack4_quantised(q[0], q[1], q[2], q[3]);
    }
}

static bool stream_dense(const NhwcGeom& g)
{
    return g.kw == 1 && g.kh == 1 && g.sw == 1 && g.sh == 1 && g.pad_top == 0 && g.pad_left == 0 && g.outw == g.W && g.outh == g.H && g.tapK == g.Cp;
}

// The tile: the smallest that gives no compute unit two (256 units), as what a tile costs is its operands' way to its unit, about 20 bytes a clock;
// larger tiles (32 x 64 to 64 x 64) were quicker nowhere.  us in a captured chain, each launch with weights of its own, the ring or the small-tile kernel /
// 16 x 16 / 16 pixels x 32 channels / 32 x 32 (one image unless said):
//   3x3 256 -> 256 on 14 x 14 7.9 / 4.1 / 5.2 / 6.4, two images 8.4 / 6.1 / 5.2 / 6.4, four 8.4 / 9.9 / 8.3 / 6.4, eight (392 tiles of 32 x 32) 8.4 / 16 / 14 / 10.4
//   1x1 1024 -> 256 on 14 x 14 5.8 / 2.7 / 3.2 / 3.7, eight images 5.8 / 8.6 / 7.5 / 5.8    1x1 2048 -> 512 on 7 x 7 7.5 / 3.8 / 4.8 / 5.8
//   3x3 512 -> 512 on 7 x 7 9.3 / 6.2 / 8.1 / 9.9, four images 9.8 / 10.0 / 8.2 / 10.1    3x3 128 -> 128 on 28 x 28 6.8 / 4.1 / 3.9 / 4.5
//   1x1 256 -> 1024 on 14 x 14, fp32 out 4.2 / 3.0 / 2.7 / 2.6    1x1 960 -> 160 on 7 x 7, fp32 out 5.2 / 2.2 / 2.7 / 3.0, 32 images 5.7 / 4.2 / 3.7 / 3.4
//   1x1 64 -> 384 on 14 x 14 2.6 / 2.1 / 2.1 / 2.3    1x1 512 -> 2048 on 7 x 7, fp32 out 4.6 / 3.0 / 2.8 / 3.2
// The limits at the short end of K are older than the loads' present order, in which a tile costs 0.5 to 1 us less, and further in than they need be: the ring is behind there too.
// Ring / here: dense on 32 x 32 tiles (56 x 56 and four images of 14 x 14) int8 out one step 2.7 / 2.4, two 2.9 / 2.4, four 3.2 and 3.8 / 2.5 against, from the line on,
// five 3.4 / 2.6; fp32 out one step 3.1 / 2.3 against two 3.3 / 2.4.  A single tap with a stride on 16 x 16 tiles int8 out one step 2.7 / 2.1, four 3.3 / 2.2 against five 3.5 / 2.2;
// fp32 out two steps 3.5 / 2.1 against three 3.6 / 2.1; on 32 x 32 int8 out seven 4.4 / 2.9 against eight 5.2 / 3.2, fp32 out five 4.5 / 2.8 against six 4.6 / 3.0.  (With two
// tiles to a unit the two are level: 64 -> 256 on 56 x 56, 784 tiles, 2.8 / 2.8, 128 -> 128 on 40 x 56, 280 tiles, 2.9 / 2.8.)
// Beyond some K the ring, which splits it over workgroups, is quicker.  Weight rows an odd number of steps (64 bytes of K) apart come in at 1.3 times the
// rate of an even number, so the lines lie further out there.  Time here over the ring's, fp32 out, dense:
//   16 x 16, below 128 tiles   even: 144 steps 0.88, 176 0.95, 192 0.94, 194 0.99, 240 1.05        odd: 401 0.75, 641 1.00, 801 1.18
//   16 x 16, from 128 on       even: 208 0.73, 240 0.86, 288 0.86-0.89, 322 0.98, 402 1.11         odd: 401 0.87, 481 0.94, 641 1.07
//   16 x 32                    even: 64 0.82, 80 0.90-0.95, 96 0.96-0.99, 112 1.12-1.14            odd: 81 0.71-0.74, 145 0.95-1.02, 193 1.07-1.12
//   32 x 32                    even: 40 0.74, 48 0.86, 56 0.97, 64 1.00, 72 1.05                   odd: 47 0.55, 49 0.74, 63 0.77
constexpr int LONGEST_32 = 48; // steps of a 32 x 32 tile
static int stream_tile(const NhwcGeom& g, int steps, bool odd, bool fp32_out, int convolutions)
{
    const long long m16 = ceil_div(g.npix, 16), m32 = ceil_div(g.npix, 32), n16 = ceil_div(g.cout, 16), n32 = ceil_div(g.cout, 32);
    const bool strided = g.ntaps == 1 && !stream_dense(g);
    if (m16 * n32 <= 256)
    {
        if (strided && steps < (fp32_out ? 3 : 5)) return 0;
        const bool wide = m16 * n16 > 256;
        const int longest = wide ? (odd ? 145 : 80) : m16 * n16 < 128 ? (odd ? 641 : 192) : (odd ? 401 : 288);
        return steps > convolutions * longest ? 0 : wide ? 12 : 11;
    }
    const int shortest = strided ? (fp32_out ? 6 : 8) : fp32_out ? 2 : 5;
    return m32 * n32 <= 256 && steps >= shortest && steps <= convolutions * LONGEST_32 ? 22 : 0;
}

// offsets are 32 bits wide and BEYOND lies beyond every buffer
static bool stream_reaches(const NhwcGeom& g)
{
    const long long limit = 1ll << 31;
    return (long long)(g.npix / (g.outw * g.outh)) * g.H * g.W * g.Cp < limit && (long long)g.cout * g.K < limit;
}

static bool stream_geometry(const NhwcGeom& g)
{
    return stream_dense(g) || (g.tapK % 64 == 0 && g.tapK == g.Cp);
}

int conv_stream_tile(const NhwcGeom& g, bool fp32_out)
{
    return stream_geometry(g) && stream_reaches(g) ? stream_tile(g, g.K / 64, g.K / 64 % 2 == 1, fp32_out, 1) : 0;
}

static int stream_tile_any_k(const NhwcGeom& g)
{
    const long long m16 = ceil_div(g.npix, 16);
    return !stream_geometry(g) ? 0 : m16 * ceil_div(g.cout, 16) <= 256 ? 11 : m16 * ceil_div(g.cout, 32) <= 256 ? 12 : 0;
}

int conv_stream_tile_any_k(const NhwcGeom& g)
{
    return stream_reaches(g) ? stream_tile_any_k(g) : 0;
}

bool conv_stream_tile_out_of_reach(const NhwcGeom& g)
{
    return stream_tile_any_k(g) != 0 && !stream_reaches(g);
}

// With a shortcut a workgroup walks both K, a round of each in flight together, in place of two launches that walk one each: the limits hold for the two together.
// us, two launches / one, main + shortcut steps: 512 channels on 7 x 7 (16 x 16 tiles) 8 + 16 5.5 / 4.1, 64 + 64 11.7 / 9.8, 192 + 192 26.1 / 24.6, 1 + 383 20.9 / 20.7; 2048 channels
// there (16 x 32) 8 + 16 6.7 / 5.0, 64 + 64 16.6 / 14.0, 80 + 80 20.1 / 18.0, 16 + 128 17.6 / 16.5; 256 channels on 28 x 28 (32 x 32) 1 + 1 6.7 / 3.5, 1 + 16 8.1 / 5.3,
// 48 + 48 16.4 / 13.8, 90 + 1 14.3 / 14.7, 1 + 90 15.0 / 14.6; beyond its limit two launches are quicker than the ring (conv_shortcut_pays).
int conv_stream_shortcut_tile(const NhwcGeom& g, int shortcut_steps)
{
    return stream_dense(g) && g.K == g.Cp && stream_reaches(g) ? stream_tile(g, g.K / 64 + shortcut_steps, g.K / 64 % 2 == 1 && shortcut_steps % 2 == 1, true, 2) : 0;
}

// where a kernel finds its last argument
template<typename Kernel>
struct LastArgument;
template<typename... Arguments>
struct LastArgument<void(Arguments...)>
{
    static constexpr size_t at()
    {
        size_t last = 0, end = 0;
        ((last = (end + alignof(Arguments) - 1) / alignof(Arguments) * alignof(Arguments), end = last + sizeof(Arguments)), ...);
        return last;
    }
};

// Steps in flight (U) and wavefronts (W) for this many steps of K: a round costs a trip to memory, and a step that only fills up a round its loads' issue.
// blocks: 16-byte operands a lane holds per step; 36 of them, 144 registers, are in flight at most.  Eight wavefronts from 49 steps on, where four would walk
// two rounds: 3x3 512 -> 512 on 7 x 7 (72 steps) 7.2 -> 6.4 us, 1x1 4096 -> 512 6.9 -> 6.0.
struct StreamForm
{
    int u, w;
};
static constexpr StreamForm stream_form(int steps, int blocks)
{
    const int w = ceil_div(steps, 4) > 12 ? 8 : 4, per_wave = ceil_div(steps, w);
    StreamForm best = {1, w};
    for (int u : {2, 4, 6, 9, 12})
        if (u * blocks <= 36 && ceil_div(per_wave, u) < ceil_div(per_wave, best.u)) best.u = u;
    return best;
}

// Whether any number of steps up to the longest that the tile meets asks for this form: only such are built.
constexpr bool stream_form_reached(int u, int w, int blocks, int longest)
{
    for (int steps = 1; steps <= longest; steps++)
    {
        const StreamForm f = stream_form(steps, blocks);
        if (f.u == u && f.w == w) return true;
    }
    return false;
}
// 32 x 32 tiles end at the limits of stream_tile (of both convolutions, which have a step each at least); beyond 1281 steps, the longest pair of the smaller ones, it is always the
// form with most in flight
constexpr int stream_longest(int tp, bool shortcut)
{
    return tp == 2 ? (shortcut ? 2 * LONGEST_32 - 1 : LONGEST_32) : 1281;
}

template<bool DENSE, int TP, int TC, int W, bool SHORTCUT>
static bool launch_stream_form(int u, const NhwcGeom& g, const int8_t* wpk, const int8_t* x, const ConvEpilogue& epi, const ConvFusion& fusion, int out_cp,
                               const StreamShortcutArg<SHORTCUT>& shortcut, hipStream_t stream)
{
    const int tiles_m = ceil_div(g.npix, 16 * TP), tiles = tiles_m * ceil_div(g.cout, 16 * TC); // 256 at most
    const int plane = g.outw * g.outh, steps = g.tapK / 64;
    const unsigned x_bytes = (unsigned)(g.npix / plane) * g.H * g.W * g.Cp;
    StreamRest<SHORTCUT> rest = {{epi.scale_in, epi.bias, epi.scale_out, fusion.residual, epi.out, fusion.q8_out, fusion.q8_scale, fusion.relu_after, epi.act}, shortcut, {}};
    if (!DENSE)
        rest.taps = {g.H, g.W, g.kw, g.dh, g.dw, g.sh, g.sw, g.pad_top, g.pad_left, g.outw, plane, steps, magic_of(plane), magic_of(g.outw), magic_of(steps), magic_of(g.kw)};
    constexpr int blocks = (TP + TC) * (SHORTCUT ? 2 : 1), longest = stream_longest(TP, SHORTCUT);
    static_assert(LastArgument<decltype(conv_stream_kernel<DENSE, TP, TC, 1, W, SHORTCUT>)>::at() == REST_AT, "`rest` lies where the kernel looks for it");
#define STREAM(U_)                                                                                                                                              \
    if constexpr (stream_form_reached(U_, W, blocks, longest))                                                                                                  \
        if (u == U_)                                                                                                                                            \
        {                                                                                                                                                       \
            const auto kernel = conv_stream_kernel<DENSE, TP, TC, U_, W, SHORTCUT>;                                                                             \
            hipLaunchKernelGGL(kernel, dim3((unsigned)tiles), dim3(64 * W), 0, stream, wpk, x, x_bytes, g.K, g.Cp, g.npix, g.cout, out_cp, tiles, tiles_m,      \
                               magic_of(tiles_m), ceil_div(g.K / 64, W), rest);                                                                                 \
            return true;                                                                                                                                        \
        }
    STREAM(1);
    STREAM(2);
    STREAM(4);
    STREAM(6);
    STREAM(9);
    STREAM(12);
#undef STREAM
    return false;
}

template<bool DENSE, bool SHORTCUT>
static int launch_stream_tile(int tile, int steps, const NhwcGeom& g, const int8_t* wpk, const int8_t* x, const ConvEpilogue& epi, const ConvFusion& fusion, int out_cp,
                               StreamShortcutArg<SHORTCUT> shortcut, hipStream_t stream)
{
    const StreamForm form = stream_form(steps, (tile / 10 + tile % 10) * (SHORTCUT ? 2 : 1));
    if constexpr (SHORTCUT) shortcut.per_wave = ceil_div(shortcut.Cp / 64, form.w);
#define STREAM_TILE(TP_, TC_)                                                                                                      \
    (form.w == 8 ? launch_stream_form<DENSE, TP_, TC_, 8, SHORTCUT>(form.u, g, wpk, x, epi, fusion, out_cp, shortcut, stream)      \
                 : launch_stream_form<DENSE, TP_, TC_, 4, SHORTCUT>(form.u, g, wpk, x, epi, fusion, out_cp, shortcut, stream))
    const bool launched = tile == 11 ? STREAM_TILE(1, 1) : tile == 12 ? STREAM_TILE(1, 2) : STREAM_TILE(2, 2);
#undef STREAM_TILE
    NCNNHIP_REQUIRE(launched, "convolution: no form of the kernel for few tiles with %d steps in flight and %d wavefronts", form.u, form.w);
    return launch_status(SHORTCUT ? "conv_stream_kernel (shortcut)" : "conv_stream_kernel");
}

int launch_conv_stream(const NhwcGeom& g, int tile, const int8_t* wpk, const int8_t* x, const ConvEpilogue& epi, const ConvFusion& fusion, int out_cp, hipStream_t stream)
{
    NCNNHIP_REQUIRE(tile && !epi.acc_out, "convolution: this layer does not fit the kernel for few tiles");
    if (stream_dense(g)) return launch_stream_tile<true, false>(tile, g.K / 64, g, wpk, x, epi, fusion, out_cp, StreamShortcutArg<false>(), stream);
    return launch_stream_tile<false, false>(tile, g.K / 64, g, wpk, x, epi, fusion, out_cp, StreamShortcutArg<false>(), stream);
}

// us, two launches / one: one image 64 + 64 -> 256 on 56 x 56 (784 tiles of 32 x 32: conv_shortcut.hip) 7.3 / 5.3, 256 + 512 -> 1024 on 14 x 14 6.4 / 4.7,
// 512 + 1024 -> 2048 on 7 x 7 6.7 / 5.0.
int launch_conv_stream_shortcut(const NhwcGeom& g, const int8_t* wpk, const int8_t* x, const ConvShortcut& sc, const ConvEpilogue& epi, const ConvFusion& fusion,
                                int out_cp, hipStream_t stream)
{
    const int tile = conv_stream_shortcut_tile(g, sc.Cp / 64);
    NCNNHIP_REQUIRE(tile && sc.Cp % 64 == 0, "convolution: this layer does not fit the kernel for few tiles");
    const int plane = sc.outw * sc.outh;
    StreamShortcutArg<true> arg;
    static_cast<ConvShortcut&>(arg) = sc;
    arg.x_bytes = (unsigned)(g.npix / plane) * sc.H * sc.W * sc.Cp;
    arg.plane = plane;
    arg.magic_plane = magic_of(plane);
    arg.magic_outw = magic_of(sc.outw);
    return launch_stream_tile<true, true>(tile, sc.Cp > g.K ? sc.Cp / 64 : g.K / 64, g, wpk, x, epi, fusion, out_cp, arg, stream);
}

} // namespace ncnnhip
