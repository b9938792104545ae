// int8 Convolution (group 1, zero border) on channels-last blobs, for layers with few output tiles: a workgroup owns 16 or 32 pixels x 16
// or 32 channels and each of its four wavefronts multiplies the whole tile over a run of K steps of its own, operands straight from
// global memory into registers in the order the matrix cores take them, 96 registers of loads in flight at once.
//
// Bound by latency: with no more tiles than compute units nothing overlaps a tile but its own loads, and the pipelined kernel
// (conv_nhwc_pipelined_kernel.h) walks K behind a barrier per 64 bytes, about 190 ns each, where here a layer is one trip to memory, a few
// dozen matrix instructions, one meeting of the sums in LDS and the epilogue.
//
// v_mfma_i32_16x16x64_i8 with weights as the A operand: a lane's four results are four neighbouring channels of one pixel, so the
// epilogue needs no transpose: four entries of each table, one 16-byte fp32 store and residual load, one 4-byte int8 store.
#include "conv_nhwc.h"

namespace ncnnhip {

typedef int v4i_cs __attribute__((ext_vector_type(4)));
typedef float v4f_cs __attribute__((ext_vector_type(4)));

// a line of zeros for operands outside the image or beyond the last K step
static __device__ __attribute__((aligned(64))) int8_t g_stream_zero_line[64];

constexpr int W = 4; // wavefronts a workgroup has

// DENSE: 1x1, stride 1, unpadded: output pixel = input pixel.  Otherwise taps of whole 64-byte steps, so that a step lies inside one tap.
// TP, TC: 16-pixel and 16-channel blocks of a tile.
// SHORTCUT: a projection shortcut is added (ConvShortcut), its K dealt out to the wavefronts and its sums met in the same way.
template<bool DENSE, int TP, int TC, bool SHORTCUT = false>
__global__ __launch_bounds__(64 * W) void conv_stream_kernel(const int8_t* __restrict__ wpk, const int8_t* __restrict__ x, NhwcGeom g, ConvEpilogue epi, ConvFusion fusion,
                                                             int out_cp, int tiles_m, unsigned magic_m, int per_wave, ConvShortcutArg<SHORTCUT> shortcut)
{
    constexpr int U = 24 / (TP + TC); // K steps a wavefront has in flight, in 96 registers
    constexpr int NB = TP * TC;     // 16 x 16 blocks of the tile
    static_assert(NB <= W, "a wavefront finishes one block");
    static_assert(!SHORTCUT || DENSE, "the sum's main convolution is 1x1");
    __shared__ v4i_cs part[SHORTCUT ? 2 : 1][W][NB][64]; // [wavefront][block][lane]
    const int lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // XCD x gets the x-th contiguous share of the tiles, the pixel tiles of one channel tile side by side: its weights cross to one XCD
    int b = blockIdx.x;
    {
        const int T = gridDim.x, xcd = b & 7, idx = b >> 3, rem = T & 7;
        b = xcd * (T >> 3) + (xcd < rem ? xcd : rem) + idx;
    }
    const int tn = tiles_m == 1 ? b : (int)__umulhi((unsigned)b, magic_m);
    const int pix0 = (b - tn * tiles_m) * (16 * TP), ch0 = tn * (16 * TC);

    const int total = g.K / 64;
    const int begin = wave * per_wave, end = begin + per_wave < total ? begin + per_wave : total;

    // wavefront q < NB finishes block q: what it needs from memory, requested before the operands (clamped addresses, nothing selected)
    const int ch4 = ch0 + wave / TP * 16 + 4 * kq, pix = pix0 + wave % TP * 16 + r16;
    float s_in[4], bias[4], s_out[4];
    float sc_in[4], sc_bias[4];
    v4f_cs res;
    const bool to_int8 = epi.scale_out != 0, with_residual = !to_int8 && fusion.residual != 0;
    if (wave < NB)
    {
        const float* bias_src = epi.bias ? epi.bias : epi.scale_in;
        const float* s_out_src = epi.scale_out ? epi.scale_out : epi.scale_in;
#pragma unroll
        for (int e = 0; e < 4; e++)
        {
            const int ch = ch4 + e < g.cout ? ch4 + e : g.cout - 1;
            s_in[e] = epi.scale_in[ch];
            bias[e] = bias_src[ch];
            s_out[e] = s_out_src[ch];
        }
        if constexpr (SHORTCUT)
        {
            const float* sc_bias_src = shortcut.bias ? shortcut.bias : shortcut.scale_in;
#pragma unroll
            for (int e = 0; e < 4; e++)
            {
                const int ch = ch4 + e < g.cout ? ch4 + e : g.cout - 1;
                sc_in[e] = shortcut.scale_in[ch];
                sc_bias[e] = sc_bias_src[ch];
            }
        }
        if (with_residual) res = *reinterpret_cast<const v4f_cs*>(fusion.residual + (size_t)(pix < g.npix ? pix : g.npix - 1) * out_cp + (ch4 < out_cp ? ch4 : out_cp - 4));
    }

    const int8_t* zero = g_stream_zero_line + kq * 16;
    const int8_t* w_row[TC];
    const int8_t* x_row[TP]; // dense: the pixel's chunk; else the pixel's image
    int iy0[TP], ix0[TP];
#pragma unroll
    for (int i = 0; i < TC; i++)
    {
        const int ch = ch0 + i * 16 + r16;
        w_row[i] = wpk + (size_t)(ch < g.cout ? ch : g.cout - 1) * g.K + kq * 16; // (a channel beyond the last: its products are not used)
    }
#pragma unroll
    for (int i = 0; i < TP; i++)
    {
        const int p = pix0 + i * 16 + r16, n = p < g.npix ? p : g.npix - 1;       // (nor are a pixel's)
        iy0[i] = ix0[i] = 0;
        if (DENSE)
            x_row[i] = x + (size_t)n * g.Cp + kq * 16;
        else
        {
            const int img = small_div(n, g.outw * g.outh), at = n - img * (g.outw * g.outh), oy = small_div(at, g.outw);
            iy0[i] = oy * g.sh - g.pad_top;
            ix0[i] = (at - oy * g.outw) * g.sw - g.pad_left;
            x_row[i] = x + (size_t)img * g.H * g.W * g.Cp + kq * 16;
        }
    }
    int tap = 0, q0 = 0, ky = 0, kx = 0; // the same in every lane
    if (!DENSE)
    {
        tap = begin * 64 / g.tapK;
        q0 = begin * 64 - tap * g.tapK;
        ky = tap / g.kw;
        kx = tap - ky * g.kw;
    }

    if constexpr (SHORTCUT)
    {
        const int8_t* sw_row[TC];
        const int8_t* sx_row[TP];
#pragma unroll
        for (int i = 0; i < TC; i++)
        {
            const int ch = ch0 + i * 16 + r16;
            sw_row[i] = shortcut.wpk + (size_t)(ch < g.cout ? ch : g.cout - 1) * shortcut.Cp + kq * 16;
        }
#pragma unroll
        for (int i = 0; i < TP; i++)
        {
            const int p = pix0 + i * 16 + r16, n = p < g.npix ? p : g.npix - 1, plane = shortcut.outw * shortcut.outh;
            const int img = small_div(n, plane), at = n - img * plane, oy = small_div(at, shortcut.outw), ox = at - oy * shortcut.outw;
            sx_row[i] = shortcut.x + (((size_t)img * shortcut.H + oy * shortcut.sh) * shortcut.W + ox * shortcut.sw) * shortcut.Cp + kq * 16;
        }
        const int steps = shortcut.Cp / 64, share = (steps + W - 1) / W;
        const int from = wave * share, to = from + share < steps ? from + share : steps;
        v4i_cs sum[NB];
#pragma unroll
        for (int q = 0; q < NB; q++) sum[q] = v4i_cs{0, 0, 0, 0};
        for (int s0 = from; s0 < to; s0 += U)
        {
            v4i_cs fw[U][TC], fx[U][TP];
#pragma unroll
            for (int u = 0; u < U; u++)
            {
#pragma unroll
                for (int i = 0; i < TC; i++) fw[u][i] = *reinterpret_cast<const v4i_cs*>(s0 + u < to ? sw_row[i] + (size_t)(s0 + u) * 64 : zero);
#pragma unroll
                for (int i = 0; i < TP; i++) fx[u][i] = *reinterpret_cast<const v4i_cs*>(s0 + u < to ? sx_row[i] + (size_t)(s0 + u) * 64 : zero);
            }
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int q = 0; q < NB; q++) sum[q] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fw[u][q / TP], fx[u][q % TP], sum[q], 0, 0, 0);
        }
#pragma unroll
        for (int q = 0; q < NB; q++) part[1][wave][q][lane] = sum[q];
    }

    v4i_cs acc[NB]; // channel block q / TP, pixel block q % TP
#pragma unroll
    for (int q = 0; q < NB; q++) acc[q] = v4i_cs{0, 0, 0, 0};
    for (int s0 = begin; s0 < end; s0 += U)
    {
        v4i_cs fw[U][TC], fx[U][TP];
#pragma unroll
        for (int u = 0; u < U; u++)
        {
            const int s = s0 + u;
            const bool live = s < end; // a step beyond the run multiplies zeros
#pragma unroll
            for (int i = 0; i < TC; i++) fw[u][i] = *reinterpret_cast<const v4i_cs*>(live ? w_row[i] + (size_t)s * 64 : zero);
#pragma unroll
            for (int i = 0; i < TP; i++)
            {
                if (DENSE)
                    fx[u][i] = *reinterpret_cast<const v4i_cs*>(live && s * 64 + kq * 16 < g.tapK ? x_row[i] + (size_t)s * 64 : zero);
                else
                {
                    const int iy = iy0[i] + ky * g.dh, ix = ix0[i] + kx * g.dw;
                    const bool in = live && tap < g.ntaps && (unsigned)iy < (unsigned)g.H && (unsigned)ix < (unsigned)g.W;
                    fx[u][i] = *reinterpret_cast<const v4i_cs*>(in ? x_row[i] + ((size_t)iy * g.W + ix) * g.Cp + q0 : zero);
                }
            }
            if (!DENSE)
            {
                q0 += 64;
                if (q0 >= g.tapK)
                {
                    q0 = 0;
                    tap++;
                    if (++kx == g.kw)
                    {
                        kx = 0;
                        ky++;
                    }
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int q = 0; q < NB; q++) acc[q] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fw[u][q / TP], fx[u][q % TP], acc[q], 0, 0, 0);
    }

    // the wavefronts' sums meet (integer addition: exact in any order)
#pragma unroll
    for (int q = 0; q < NB; q++) part[0][wave][q][lane] = acc[q];
    __syncthreads();
    if (wave >= NB || ch4 >= out_cp || pix >= g.npix) return;
    v4i_cs sum = part[0][0][wave][lane];
#pragma unroll
    for (int s = 1; s < W; s++) sum += part[0][s][wave][lane];

    // the pipelined kernel's epilogue, statement by statement
    float f[4];
#pragma unroll
    for (int e = 0; e < 4; e++)
    {
        f[e] = mul_rn((float)sum[e], s_in[e]);
        f[e] = add_rn(f[e], epi.bias ? bias[e] : -0.f); // no bias: -0, the one value whose addition changes nothing
    }
    if (epi.act.type == 1)
    {
#pragma unroll
        for (int e = 0; e < 4; e++) f[e] = fmaxf(f[e], 0.f);
    }
    else if (epi.act.type != 0)
    {
#pragma unroll
        for (int e = 0; e < 4; e++) f[e] = apply_activation(f[e], epi.act);
    }
    const size_t o = (size_t)pix * out_cp + ch4;
    if (to_int8)
    {
#pragma unroll
        for (int e = 0; e < 4; e++) f[e] = mul_rn(f[e], s_out[e]);
        float2int8_as_float_x4(f[0], f[1], f[2], f[3]);
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (ch4 + e >= g.cout) f[e] = 0.f; // channels from cout up to out_cp are the blob's zero padding
        *reinterpret_cast<uint32_t*>(static_cast<int8_t*>(epi.out) + o) = pack4_quantised(f[0], f[1], f[2], f[3]);
        return;
    }
    v4f_cs v;
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = ch4 + e < g.cout ? f[e] : 0.f;
    if constexpr (SHORTCUT)
    {
        v4i_cs other = part[1][0][wave][lane];
#pragma unroll
        for (int s = 1; s < W; s++) other += part[1][s][wave][lane];
#pragma unroll
        for (int e = 0; e < 4; e++)
        {
            float t = add_rn(mul_rn((float)other[e], sc_in[e]), shortcut.bias ? sc_bias[e] : -0.f);
            if (shortcut.act.type != 0) t = apply_activation(t, shortcut.act);
            v[e] = add_rn(v[e], ch4 + e < g.cout ? t : 0.f);
        }
    }
    if (with_residual)
    {
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = add_rn(v[e], res[e]);
    }
    if (fusion.relu_after)
    {
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = v[e] < 0.f ? 0.f : v[e]; // the ReLU LAYER's statement (src/layer/relu.cpp:36-37): a NaN stays, unlike fmaxf
    }
    if (epi.out) *reinterpret_cast<v4f_cs*>(static_cast<float*>(epi.out) + o) = v;
    if (fusion.q8_out)
    {
        float q[4];
#pragma unroll
        for (int e = 0; e < 4; e++) q[e] = mul_rn(v[e], fusion.q8_scale);
        float2int8_as_float_x4(q[0], q[1], q[2], q[3]);
        *reinterpret_cast<uint32_t*>(fusion.q8_out + o) = pack4_quantised(q[0], q[1], q[2], q[3]);
    }
}

static bool stream_dense(const NhwcGeom& g)
{
    return g.kw == 1 && g.kh == 1 && g.sw == 1 && g.sh == 1 && g.pad_top == 0 && g.pad_left == 0 && g.outw == g.W && g.outh == g.H && g.tapK == g.Cp;
}

// The tile: the smallest that gives no compute unit two (256 units), as what a tile costs is its operands' way to its unit, about 20 bytes a clock;
// larger tiles (32 x 64 to 64 x 64) were quicker nowhere.  us in a captured chain, weights from HBM, the small-tile or pipelined kernel /
// 16 x 16 / 16 pixels x 32 channels / 32 x 32 (56 x 56 to 7 x 7, one image unless said):
//   3x3 256 -> 256 on 14 x 14 8.5 / 4.7 / 6.1 / 7.2, two images 8.6 / 6.8 / 6.1 / 7.2, four 8.6 / 10.8 / 9.6 / 7.3, eight (392 tiles of 32 x 32) 8.7 / 17 / 17 / 11.4
//   1x1 1024 -> 256 on 14 x 14 5.8 / 3.7 / 4.1 / 4.7, eight images 6.0 / 11.6 / 9.0 / 6.7    1x1 2048 -> 512 on 7 x 7 7.4 / 4.9 / 5.6 / 7.2
//   3x3 512 -> 512 on 7 x 7 9.9 / 7.0 / 9.2 / 10.7    3x3 128 -> 128 on 28 x 28 6.9 / 5.4 / 4.4 / 5.2    1x1 256 -> 1024 on 14 x 14, fp32 out 5.0 / 6.0 / 4.5 / 4.1
//   1x1 960 -> 160 on 7 x 7, fp32 out 5.0 / 3.4 / 3.6 / 4.0, 32 images 6.0 / 6.7 / 5.1 / 4.6    1x1 64 -> 384 on 14 x 14 3.0 / 2.9 / 2.9 / 3.2
// With 32 x 32 tiles the ring is level or ahead at both ends of K: int8 out 1x1 64 -> 64 on 56 x 56 3.0 / 3.2, 256 -> 64 3.6 / 3.9, 3x3 512 -> 512 on 7 x 7,
// eight images 10.7 / 11.0 (four, 16 x 32 tiles: 10.2 / 9.2); fp32 out is ahead from two steps on (128 -> 64 on 56 x 56 3.34 / 3.21, 192 -> 64 3.52 / 3.31,
// 256 -> 64 level, 3.68 / 3.71).
// A single tap with a stride (1x1, not dense) costs its pixels' divisions and, on the ring, no more than a dense one: the ring is ahead of the smaller tiles below
// five steps to int8 (64 -> 256 on 28 x 28, stride 2, 3.1 / 3.8; 256 -> 256 3.6 / 3.7, 320 -> 256 3.8 / 3.6) and three to fp32 (128 3.5 / 3.6, 192 3.6 / 3.6), of
// 32 x 32 below eight and six (four images, int8 384 4.0 / 4.1, 512 5.3 / 4.5; fp32 256 3.9 / 4.2, 384 4.2 / 4.1).
// Beyond some K the ring, which splits it over workgroups, is quicker again.  Weight rows an odd number of steps (64 bytes of K) apart come in at 1.3 times the
// rate of an even number, so the lines lie further out there.  Time here over the ring's, fp32 out, dense:
//   16 x 16, below 128 tiles   even: 144 steps 0.87-0.93, 176 0.94-0.99, 194 1.00-1.06, 288 1.03-1.09    odd: 193 0.8, 401 0.86-0.91, 641 0.88-0.95
//   16 x 16, from 128 on       even: 208 0.81-0.93, 288 0.91-0.98, 322 0.98-1.08, 402 1.02-1.23          odd: 401 0.78-0.94, 641 1.09-1.20
//   16 x 32                    even: 64 0.87-0.91, 80 0.96-1.02, 96 1.04-1.05, 144 1.2, 402 2.0          odd: 81 0.8, 145 0.92-1.00, 193 1.00-1.17
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
    return m32 * n32 <= 256 && steps >= shortest && steps <= convolutions * 48 ? 22 : 0;
}

static bool stream_addressing(const NhwcGeom& g)
{
    return stream_dense(g) || (g.tapK % 64 == 0 && g.tapK == g.Cp);
}

int conv_stream_tile(const NhwcGeom& g, bool fp32_out)
{
    return stream_addressing(g) ? stream_tile(g, g.K / 64, g.K / 64 % 2 == 1, fp32_out, 1) : 0;
}

int conv_stream_tile_any_k(const NhwcGeom& g)
{
    const long long m16 = ceil_div(g.npix, 16);
    return !stream_addressing(g) ? 0 : m16 * ceil_div(g.cout, 16) <= 256 ? 11 : m16 * ceil_div(g.cout, 32) <= 256 ? 12 : 0;
}

// With a shortcut a workgroup walks both K, one after the other, in place of two launches that walk one each: the limits hold for the two together.
// us, two launches / one, main + shortcut steps: 512 channels on 7 x 7 (16 x 16 tiles) 8 + 16 7.6 / 5.8, 64 + 64 13.6 / 11.7, 100 + 100 18.4 / 16.3; 2048 channels
// there (16 x 32) 8 + 16 8.9 / 6.9, 64 + 64 18.6 / 16.6; 256 channels on 28 x 28 (32 x 32) 1 + 1 7.2 / 4.5 (the ring: 5.0), 1 + 16 9.0 / 6.2 (10.0),
// 48 + 48 17.7 / 15.5, 64 + 32 17.3 / 16.5 (35.8); beyond its limit two launches are quicker than the ring (conv_shortcut_pays).
int conv_stream_shortcut_tile(const NhwcGeom& g, int shortcut_steps)
{
    return stream_dense(g) && g.K == g.Cp ? stream_tile(g, g.K / 64 + shortcut_steps, g.K / 64 % 2 == 1 && shortcut_steps % 2 == 1, true, 2) : 0;
}

int launch_conv_stream(const NhwcGeom& g, int tile, const int8_t* wpk, const int8_t* x, const ConvEpilogue& epi, const ConvFusion& fusion, int out_cp, hipStream_t stream)
{
    const int tp = tile / 10, tc = tile % 10;
    NCNNHIP_REQUIRE(tile && !epi.acc_out, "convolution: this layer does not fit the kernel for few tiles");
    const int tiles_m = ceil_div(g.npix, 16 * tp), tiles_n = ceil_div(g.cout, 16 * tc), blocks = tiles_m * tiles_n; // 256 at most
    const unsigned magic_m = tiles_m > 1 ? (unsigned)((1ull << 32) / (unsigned)tiles_m + 1) : 0u;
    const int per_wave = ceil_div(g.K / 64, W);
#define STREAM(DENSE_, TP_, TC_)                                                                                                                            \
    hipLaunchKernelGGL((conv_stream_kernel<DENSE_, TP_, TC_>), dim3((unsigned)blocks), dim3(64 * W), 0, stream, wpk, x, g, epi, fusion, out_cp, tiles_m, magic_m, \
                       per_wave, ConvShortcutArg<false>())
#define STREAM_TILE(DENSE_)       \
    do                            \
    {                             \
        if (tile == 11)           \
            STREAM(DENSE_, 1, 1); \
        else if (tile == 12)      \
            STREAM(DENSE_, 1, 2); \
        else                      \
            STREAM(DENSE_, 2, 2); \
    } while (0)
    if (stream_dense(g))
        STREAM_TILE(true);
    else
        STREAM_TILE(false);
#undef STREAM_TILE
#undef STREAM
    return launch_status("conv_stream_kernel");
}

// us, two launches / one: one image 64 + 64 -> 256 on 56 x 56 (784 tiles of 32 x 32: conv_shortcut.hip) 8.0 / 5.5, 256 + 512 -> 1024 on 14 x 14 8.4 / 6.4,
// 512 + 1024 -> 2048 on 7 x 7 8.0 / 6.3.
int launch_conv_stream_shortcut(const NhwcGeom& g, const int8_t* wpk, const int8_t* x, const ConvShortcut& sc, const ConvEpilogue& epi, const ConvFusion& fusion,
                                int out_cp, hipStream_t stream)
{
    const int tile = conv_stream_shortcut_tile(g, sc.Cp / 64), tp = tile / 10, tc = tile % 10;
    NCNNHIP_REQUIRE(tile && sc.Cp % 64 == 0, "convolution: this layer does not fit the kernel for few tiles");
    const int tiles_m = ceil_div(g.npix, 16 * tp), tiles_n = ceil_div(g.cout, 16 * tc);
    const unsigned magic_m = tiles_m > 1 ? (unsigned)((1ull << 32) / (unsigned)tiles_m + 1) : 0u;
    ConvShortcutArg<true> arg;
    static_cast<ConvShortcut&>(arg) = sc;
#define STREAM(TP_, TC_)                                                                                                                                               \
    hipLaunchKernelGGL((conv_stream_kernel<true, TP_, TC_, true>), dim3((unsigned)(tiles_m * tiles_n)), dim3(64 * W), 0, stream, wpk, x, g, epi, fusion, out_cp, tiles_m, \
                       magic_m, ceil_div(g.K / 64, W), arg)
    if (tile == 11)
        STREAM(1, 1);
    else if (tile == 12)
        STREAM(1, 2);
    else
        STREAM(2, 2);
#undef STREAM
    return launch_status("conv_stream_kernel (shortcut)");
}

} // namespace ncnnhip
