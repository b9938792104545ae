// The pipelined channels-last convolution kernel's launches with one workgroup per output tile: Convolution (every
// addressing mode) and InnerProduct, the planner they share with the other forms, and the InnerProduct entry that
// allocates nothing.  The kernel itself is in conv_nhwc_pipelined_kernel.h.
#include "conv_nhwc_pipelined_kernel.h"

namespace ncnnhip {

constexpr int SPLIT_MIN_STEPS = 12;

PipePlan plan_pipelined(int cout, long long npix, int steps)
{
    PipePlan p;
    p.groups = 1;
    // (A layer whose K stays whole in four wavefronts takes choose_tile's instead.)  Channel tile: the width that pads the channel count least (padded channels cost matrix-core time and unbalance the
    // wavefronts' epilogues: 144 channels in one 256-wide tile ran 34 us, in three 64-wide tiles 21), the wider on a tie
    p.bn = 64;
    for (int bn = 128; bn <= 256; bn *= 2)
        if (ceil_div(cout, bn) * bn <= ceil_div(cout, p.bn) * p.bn) p.bn = bn;
    p.bm = 128;
    auto tiles = [&]() { return (long long)ceil_div(npix, p.bm) * ceil_div(cout, p.bn); };
    // measured over the ResNet-50 / MobileNetV2 layers: more, smaller workgroups win until there are a few
    // thousand of them (these layers are latency bound, not matrix-core bound)
    if (tiles() < 100000) p.bm = 64;
    if (tiles() < 1024 && p.bn == 256) p.bn = 128;
    if (tiles() < 512 && p.bn == 128 && cout > 64) p.bn = 64;
    p.tiles_m = ceil_div(npix, p.bm);
    p.tiles_n = ceil_div(cout, p.bn);
    p.splits = 1;
    const long long t = tiles();
    if (t < 256 && t <= SPLIT_MAX_TILES && steps >= 2 * SPLIT_MIN_STEPS)
    {
        // fewer tiles than CUs: split K until there is about one workgroup per CU (two splits from 128 tiles up; with the
        // limit at 128 tiles the 196-tile 3x3 layers of ResNet-50's fourth stage at batch 16 ran unsplit on 196 of the 256
        // CUs), at least 12 steps each.  A split costs about 2 us (partial sums through memory, the last workgroup of a
        // tile adds them up): with 8 steps each, the 16-step 1x1 layers 1024 -> 256 of ResNet-50 ran 8.6 us in two halves
        // and 6.8 whole at batch 16, the 18-step 3x3 layers 128 -> 128 9.6 and 7.5 at batch 8; summed over a pass the
        // kernels take 350 / 355 / 362 / 385 us at batch 1 with at least 8 / 12 / 16 / 24 steps, 404 / 389 / 395 / 414
        // at batch 4, 459 / 449 / 446 / 466 at batch 8, 568 / 555 / 556 / 565 at batch 16 (MobileNetV2: no difference).
        // (The int8 layers of those passes with few small tiles have gone to conv_stream_kernel since; here still come InnerProduct,
        // the loader of fp32 and fp16 blobs, taps that are no whole steps, a K too long for that kernel, and more tiles than it takes.)
        const int want = (int)((256 + t - 1) / t);
        const int max_splits = steps / SPLIT_MIN_STEPS;
        p.splits = want < max_splits ? want : max_splits;
        if (p.splits < 1) p.splits = 1;
    }
    p.steps_per_split = ceil_div(steps, p.splits);
    p.splits = ceil_div(steps, p.steps_per_split);
    return p;
}

PipePlan plan_pipelined_groups(int cout, long long npix, int steps)
{
    PipePlan p = plan_pipelined(cout, npix, steps);
    const long long t = (long long)p.tiles_m * p.tiles_n;
    // With no more tiles than compute units a 64 x 64 tile has a unit to itself, and four wavefronts there wait for each K
    // step's loads in turn; sixteen have four steps under way.  us, four wavefronts -> sixteen, one layer alone:
    //   1x1 1024 -> 256 on 14x14: batch 1 6.3 -> 5.6, batch 16 6.5 -> 5.9    1x1 2048 -> 512 on 7x7: 8.2 -> 7.2, batch 16 9.3 -> 7.4
    //   1x1 960 -> 160 on 7x7 6.0 -> 5.2    3x3 256 -> 256 on 14x14, batch 16 11.4 -> 8.7    3x3 512 -> 512 on 7x7, batch 16 12.7 -> 11.5
    // Eight wavefronts gain about half of that.  The lines, from 1x1 and 3x3 layers of 8 to 100 steps on 2 to 441 tiles:
    // (of these the batch-1 layers and 960 -> 160 run on conv_stream_kernel by now.)
    //   beyond 256 tiles two of them share a unit and sixteen lose: 24 steps, 196 tiles 10.1 -> 7.2, 320 tiles 9.1 -> 12.2; 72 steps
    //   196 tiles 16.2 -> 13.5, 320 tiles 20.9 -> 24.6;
    //   with 8 and 9 steps they are up to 3 % slower alone (75 tiles 4.76 -> 4.84 and 4.94 -> 5.05), from 11 on faster (5.55 -> 5.42 at
    //   12); the nets' passes, which have those layers too, were no slower with them.
    if (p.bm != 64 || p.bn != 64 || steps < 8 || t > 256) return p;
    // A few tiles of a long K want other compute units more than wavefronts of their own.  Four wavefronts in splits / sixteen in one:
    // (InnerProduct, steps that meet several taps, a K beyond conv_stream_kernel's) 3x3 of 36 steps 16 tiles 8.2 / 8.5, 52 tiles 8.9 / 8.7; 45 steps 20 tiles 8.8 / 9.6.  (From 72 steps on three splits of sixteen
    // would be better still: 20 tiles 10.4 -> 10.1, 1x1 of 100 steps 12.0 -> 10.4.)
    if (p.splits >= 3 && t < 24) return p;
    p.groups = 4;
    // K is split over workgroups as well while they fit the chip, at least 24 steps each: 512 -> 512 on 7x7, batch 4 (32 tiles)
    // 11.0 in six splits of four wavefronts, 10.1 in three of sixteen, 10.8 in four; 1x1 of 100 steps, 52 tiles 14.9 / 12.0 / 11.1 / 11.7
    // in one to four.  Up to 40 tiles two halves pay from 40 steps on: 3x3 of 41 steps, 28 tiles 9.7 in one, 8.8 in two (9.0 in three
    // splits of four wavefronts), 1x1 of 46 steps 8.9 and 8.7; with 64 tiles 9.8 and 9.4, 9.2 and 9.3.
    const int room = (int)(256 / t);
    int longest = steps / 24;
    if (longest < 2 && steps >= 40 && t <= 40) longest = 2;
    p.splits = std::max(1, std::min(p.splits, std::min(room, longest)));
    p.steps_per_split = ceil_div(steps, p.splits);
    p.splits = ceil_div(steps, p.steps_per_split);
    return p;
}

size_t conv_nhwc_pipelined_workspace_words(int cout, long long npix, int steps)
{
    const PipePlan p = plan_pipelined(cout, npix, steps);
    if (p.splits <= 1) return 0;
    return SPLIT_COUNTER_BYTES / sizeof(int32_t) + (size_t)p.splits * p.tiles_m * p.tiles_n * p.bm * p.bn;
}

static int special_kernel(const NhwcGeom& g, const ConvEpilogue& epi, const ConvFusion& fusion, int out_cp)
{
    if (conv_pointwise_fits(g, epi, fusion, out_cp) || conv_pointwise_stem_fits(g, epi, fusion, out_cp)) return NCNNHIP_CONV_POINTWISE;
    if (conv_resident_fits(g, epi, fusion, out_cp)) return NCNNHIP_CONV_RESIDENT;
    return conv_stream_tile(g, !epi.scale_out) ? NCNNHIP_CONV_FEW_TILES : NCNNHIP_CONV_PIPELINED;
}

// The tile of a layer whose K stays whole in four wavefronts.  A unit holds five workgroups of 64 x 64 pixels x channels, three of 64 x 128, two of 128 x 128; a wide tile reads half as much
// from LDS for a product, and computes a pixel's address (a division, where the layer has taps or a stride) for twice the channels.  Measured in captured chains and in passes of ResNet-50 and MobileNetV2.
//   64 x 128 over 64 x 64, by tiles of 64 x 128 (256 to 2048 channels): 384, where 64 x 64 are three to a unit, 16 and 18 steps 1.09 to 1.11, 36 1.05, 10 to 14 1.10 to 1.14, 3x3 to int8 5 1.09, 12
//   and 14 1.01; from 400 on, where these are four: 16 and 18 steps 0.94 to 1.00, 23 and 36 0.79 to 0.91, 10 to 14 to int8 0.91 to 1.02, 3x3 to int8 5 0.93 to 1.01, 9 to 14 0.87 to 0.97, 3x3 to fp32 12 and 14
//   0.91 to 1.02; with fewer steps, to fp32 or of a sum only beyond five to a unit (640): 10 and 14 steps to fp32 576 and 608 1.02 to 1.05, 688 0.96 to 1.01, 8 to int8 608 0.98 to 1.01, 688 0.91
//   to 0.94, sums of 16 and 18 608 1.05, 688 0.92 to 0.94 (1040 1.06 to 1.08, 1200 0.97: between 1024 and 1160 they stay with 64 x 64), 3x3 of four to nine steps to fp32 676 0.94 to 0.96; with a short K beyond 900:
//   one step 25088 x 384 7.5 8.6 us, 12544 x 384 5.1 6.0 (one tile for all channels is left as wide as they are), two 12544 x 576 7.6 6.9, four and five 100352 x 128 14.4 13.9, 6272 x 1280 14.2
//   13.0; to int8 from 700 with a stride, one step 784 tiles 6.8 6.6, 1568 10.5 10.1, 1536 10.5 9.7 (500 tiles 4.7 4.8; to fp32 784 tiles 8.5 8.3, 1568 the other way by 4 to 8 %), and from 750
//   where the one tile for all channels is partly padding, 96 channels 784 tiles 5.7 5.6, 896 6.0 5.8 (128 channels 784 tiles level).
//   128 x 128 over 64 x 128, by tiles of 128 x 128: 384 of them 8 to 18 steps 1.00 to 1.13, 392, where 64 x 128 ones are more than three to a unit, 0.80 to 0.95 (8 steps to fp32 0.98 to 1.00, with
//   64 x 64 the quickest); earlier from 300 with 23 steps and more, 304 0.93 to 1.04, 344 0.89 to 1.01 (a sum 1.00 to 1.04), or to int8 and more than 128 channels with 16, dense 304 0.99, 344 0.96, 3x3
//   344 1.03, 368 1.00.  Beyond the 512 that are one round it is behind, 528 16 to 23 steps 1.08 to 1.15, 640 1.02 to 1.13, until 670, 680 0.94 to 1.07, 720 0.93 to 1.09 (to fp32 with 16
//   and 18 until 770, 680 1.04 to 1.07, 768 1.02 and 1.04, 784 0.95 to 1.02; of a sum of 23 until 850, 640 1.17, 832 1.02, 900 0.94); with 9 to 15 steps at 784 0.95 to 1.18, and with 10 ahead again at 2256, 0.88 to
//   1.00; a sum of 18 steps at 784 1.05.  25088 x 256, us of the three, 36 steps 35.6 32.6 23.6, 16 19.2 18.9 15.8, 8 12.6 13.0 12.0; sums 6272 x 1024, 36 steps 37.4 36.9 28.8, 12544 x 1024 69 62 56.
//   A sum (residual in, fp32 and int8 out) of a short K is bound by memory, and small tiles keep more of it in flight: 64 x 64 / 64 x 128 50176 x 512 24.8 27.0, 25088 x 1024 29.7 31.0, 25088 x 512 15.0 16.8,
//   6272 x 1024 10.8 12.3, 50176 x 256 14.3 16.1, 12544 x 1024 21.6 22.5; from about 7000 of them on, where its blobs no longer stay in the 256 MB in front of HBM, 64 x 128 is as good or better: 6656 tiles, 26624 x
//   1024, two to four steps 37.5 to 40.4 / 37.4 to 41.2, 7168 47.9 46.5 to 61.1 56.5, 7680 56.9 52.6 to 69.4 60.7; 401408 x 256 112.7 104.8, 100352 x 512 93.0 87.1; with 8 steps from 3000: 6272 x 2048 31.2 30.2.
// (64 x 256 is the best nowhere, 128 x 64 where 64 x 128 is nearly as good.)
static void choose_tile(const NhwcGeom& g, bool residual, bool int8_out, bool dense, PipePlan& p)
{
    const int steps = g.K / 64;
    const auto tiles = [&](int bm, int bn) { return (long long)ceil_div(g.npix, bm) * ceil_div(g.cout, bn); };
    const bool wide = ceil_div(g.cout, 128) * 128 <= ceil_div(g.cout, 64) * 64; // without more padded channels
    const bool taps = g.ntaps > 1;
    const long long t64 = tiles(64, 64), t128 = tiles(64, 128), square = tiles(128, 128);
    p.bm = p.bn = 64;
    if (residual && steps < 14)
    {
        if (wide && t64 >= (steps >= 8 ? 3000 : 7000)) p.bn = 128;
    }
    else if (wide)
    {
        const long long first = steps < 16 || residual ? 385 : steps >= 23 ? 300 : int8_out && g.cout > 128 ? (dense ? 300 : 360) : 385;
        const long long again = residual ? 850 : steps < 16 ? 2000 : !int8_out && steps < 20 ? 770 : 670;
        const bool square_pays = steps >= (int8_out ? 8 : 10) && square >= first && (square <= 512 || (square > again && steps >= (residual ? 23 : 10)));
        const bool four_to_a_unit = residual ? steps >= 23 : steps >= 16 || (int8_out && (steps >= 10 || (taps && steps >= 5))) || (taps && steps >= 12);
        const bool six_to_a_unit = taps || steps >= 14 || (int8_out && steps >= 8);
        if (square_pays)
            p.bm = p.bn = 128;
        else if (t128 > (four_to_a_unit ? 384 : six_to_a_unit ? 640 : 899) && (steps >= 2 || g.cout <= 128))
            p.bn = residual && steps < 23 && t128 > 1024 && t128 < 1160 ? 64 : 128;
        else if (int8_out && ((!dense && t128 >= 700) || (g.cout < 128 && t128 >= 750)))
            p.bn = 128;
    }
    if (!tiles_fit_a_launch(ceil_div(g.npix, 64), ceil_div(g.cout, p.bn))) // (an output of 69 GB and more)
    {
        p.bm = 128;
        p.bn = wide ? 128 : 64;
        if (!tiles_fit_a_launch(ceil_div(g.npix, 128), ceil_div(g.cout, p.bn)) && ceil_div(g.cout, 256) * 256 <= ceil_div(g.cout, p.bn) * p.bn) p.bn = 256;
    }
    p.tiles_m = ceil_div(g.npix, p.bm);
    p.tiles_n = ceil_div(g.cout, p.bn);
}

// the pipelined kernel's plan and addressing mode (its MODE), the layer as it sees it in g
static int pipelined_form(NhwcGeom& g, const ConvEpilogue& epi, const ConvFusion& fusion, PipePlan& p)
{
    // A 1x1, stride-1, unpadded layer reads input pixel n for output pixel n, whatever the image shape: present it as
    // one row of npix pixels, and the kernel skips the pixel -> (image, y, x) divisions.
    const int dense = g.kw == 1 && g.kh == 1 && g.sw == 1 && g.sh == 1 && g.pad_top == 0 && g.pad_left == 0 && g.outw == g.W && g.outh == g.H && g.tapK == g.Cp;
    if (dense)
    {
        g.H = g.outh = 1;
        g.W = g.outw = g.npix;
    }
    p = plan_pipelined_groups(g.cout, g.npix, g.K / 64);
    if (p.groups == 1 && p.splits == 1) choose_tile(g, fusion.residual != 0, epi.scale_out != 0, dense, p);
    // the narrow-input first layer has four K steps at most: from a million output pixels up, 128-pixel tiles halve the number of
    // workgroup prologues (ResNet-50's 7 x 7 first layer at batch 128: the pass 2.22 -> 2.20 ms; at batch 16, 0.2 M pixels, no gain)
    if ((g.tapK == 16 || g.tapK == 32) && p.splits == 1 && p.bm == 64 && g.npix >= (1 << 20))
    {
        p.bm = 128;
        p.tiles_m = ceil_div(g.npix, 128);
    }
    // (the K-split kernels exist for modes 0, 1 and 3 only: a narrow-input layer has too few K steps to be split)
    return dense ? 1 : (p.groups == 1 && (g.tapK == 16 || g.tapK == 32) && p.splits == 1) ? 2 : (g.tapK % 64 == 0 && g.tapK == g.Cp) ? 3 : 0;
}

void conv_nhwc_pipelined_route(const NhwcGeom& g_in, const ConvEpilogue& epi, const ConvFusion& fusion, int out_cp, ncnnhip_conv_route& route)
{
    route = {special_kernel(g_in, epi, fusion, out_cp), 0, 0, 0, 0, 0};
    if (route.kernel == NCNNHIP_CONV_FEW_TILES)
    {
        const int tile = conv_stream_tile(g_in, !epi.scale_out);
        route.tile_pixels = tile / 10 * 16;
        route.tile_channels = tile % 10 * 16;
    }
    if (route.kernel != NCNNHIP_CONV_PIPELINED) return;
    NhwcGeom g = g_in;
    PipePlan p;
    const int mode = pipelined_form(g, epi, fusion, p);
    route = {NCNNHIP_CONV_PIPELINED, p.bm, p.bn, mode, p.groups, p.splits};
}

int launch_conv_nhwc_pipelined(const NhwcGeom& g_in, const int8_t* wpk, const int8_t* x, const ConvEpilogue& epi, const ConvFusion& fusion, int out_cp,
                               void* workspace, size_t workspace_bytes, hipStream_t stream)
{
    switch (special_kernel(g_in, epi, fusion, out_cp))
    {
    case NCNNHIP_CONV_POINTWISE:
        return launch_conv_pointwise(g_in, wpk, x, epi, out_cp, stream);
    case NCNNHIP_CONV_RESIDENT:
        return launch_conv_resident(g_in, wpk, x, epi, fusion, out_cp, stream);
    case NCNNHIP_CONV_FEW_TILES:
        return launch_conv_stream(g_in, conv_stream_tile(g_in, !epi.scale_out), wpk, x, epi, fusion, out_cp, stream);
    }
    NhwcGeom g = g_in;
    PipePlan p;
    const int mode = pipelined_form(g, epi, fusion, p);
    NCNNHIP_REQUIRE(tiles_fit_a_launch(p.tiles_m, p.tiles_n), "convolution: too many tiles"); // (a K split is of 256 tiles at most)
    int32_t* partial = 0;
    unsigned* counters = 0;
    if (p.splits > 1)
    {
        const size_t need = SPLIT_COUNTER_BYTES + (size_t)p.splits * p.tiles_m * p.tiles_n * p.bm * p.bn * sizeof(int32_t);
        const bool split = workspace && workspace_bytes >= need;
        const int tile = split ? 0 : conv_stream_tile_any_k(g_in);
        if (tile) return launch_conv_stream(g_in, tile, wpk, x, epi, fusion, out_cp, stream);
        if (!split && conv_stream_tile_out_of_reach(g_in))
            p.splits = 1; // (an input of 2 GiB under a few tiles: K stays whole)
        else
        {
            NCNNHIP_REQUIRE(split, "convolution: workspace of %zu bytes required", need);
            counters = (unsigned*)workspace; // zero on entry (the caller cleared the workspace once), zero again on exit
            partial = (int32_t*)((char*)workspace + SPLIT_COUNTER_BYTES);
        }
    }
    dim3 grid((unsigned)((long long)p.tiles_m * p.tiles_n * p.splits)), block((unsigned)(256 * p.groups));
    if (p.splits > 1) return launch_pipe_split(p, mode, wpk, x, g, epi, fusion, out_cp, out_cp, partial, counters, stream);
#define LAUNCH_PIPE_MODE(BM_, BN_, MODE_, GROUPS_)                                                                                                                 \
    hipLaunchKernelGGL((conv_nhwc_pipelined_kernel<BM_, BN_, PIPE_RING, false, MODE_, 1, GROUPS_>), grid, block, 0, stream, wpk, x, g, epi, fusion, out_cp, \
                       out_cp, p.tiles_m, p.tiles_n, p.splits, p.steps_per_split, tile_magic(p.tiles_n), partial, counters, (const float*)0, 0, ConvShortcutArg<false>())
#define LAUNCH_PIPE(BM_, BN_)                  \
    do                                         \
    {                                          \
        if (mode == 1)                         \
            LAUNCH_PIPE_MODE(BM_, BN_, 1, 1);  \
        else if (mode == 2)                    \
            LAUNCH_PIPE_MODE(BM_, BN_, 2, 1);  \
        else if (mode == 3)                    \
            LAUNCH_PIPE_MODE(BM_, BN_, 3, 1);  \
        else                                   \
            LAUNCH_PIPE_MODE(BM_, BN_, 0, 1);  \
    } while (0)
    if (p.groups == 4 && mode == 1)
        LAUNCH_PIPE_MODE(64, 64, 1, 4);
    else if (p.groups == 4 && mode == 3)
        LAUNCH_PIPE_MODE(64, 64, 3, 4);
    else if (p.groups == 4)
        LAUNCH_PIPE_MODE(64, 64, 0, 4);
    else if (p.bm == 128 && p.bn == 256)
        LAUNCH_PIPE(128, 256);
    else if (p.bm == 128 && p.bn == 128)
        LAUNCH_PIPE(128, 128);
    else if (p.bm == 128) // narrow inputs, and more tiles than a launch holds
        LAUNCH_PIPE(128, 64);
    else if (p.bn == 128)
        LAUNCH_PIPE(64, 128);
    else
        LAUNCH_PIPE(64, 64);
#undef LAUNCH_PIPE
#undef LAUNCH_PIPE_MODE
    return launch_status("conv_nhwc_pipelined_kernel");
}

int launch_fc_via_conv_pipelined(const int8_t* x, size_t x_stride, int rows, int K, int num_output, const int8_t* weight, const ConvEpilogue& epi,
                                 size_t out_stride, void* workspace, size_t workspace_bytes, hipStream_t stream, bool* handled)
{
    *handled = false;
    const bool aligned = ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(weight) | reinterpret_cast<uintptr_t>(epi.out)) & 15) == 0;
    if (K % 64 || num_output % 4 || x_stride % 16 || out_stride % 4 || !aligned || epi.scale_out || epi.acc_out) return NCNNHIP_OK;
    if ((long long)rows * (long long)x_stride >= (1ll << 31)) return NCNNHIP_OK;
    const size_t need = conv_nhwc_pipelined_workspace_words(num_output, rows, K / 64) * sizeof(int32_t);
    if (need > workspace_bytes || (need && !workspace)) return NCNNHIP_OK;
    *handled = true;

    NhwcGeom g;
    g.H = 1;
    g.W = rows;
    g.Cp = (int)x_stride;
    g.tapK = g.Cp;
    g.kw = g.kh = g.dw = g.dh = g.sw = g.sh = 1;
    g.pad_top = g.pad_left = 0;
    g.outw = rows;
    g.outh = 1;
    g.npix = rows;
    g.ntaps = 1;
    g.K = K;
    g.cout = num_output;
    g.pad_word = 0;
    const ConvFusion no_fusion = {0, 0, 0, 0.f};
    const PipePlan p = plan_pipelined_groups(num_output, rows, K / 64);
    int32_t* partial = 0;
    unsigned* counters = 0;
    if (p.splits > 1)
    {
        counters = (unsigned*)workspace;
        partial = (int32_t*)((char*)workspace + SPLIT_COUNTER_BYTES);
    }
    NCNNHIP_REQUIRE((long long)p.tiles_m * p.tiles_n * p.splits * p.tiles_n < (1ll << 32), "innerproduct: too many tiles");
    dim3 grid((unsigned)((long long)p.tiles_m * p.tiles_n * p.splits)), block((unsigned)(256 * p.groups));
    // rows are few: only the 64-pixel tiles occur
    if (p.bm != 64)
    {
        *handled = false;
        return NCNNHIP_OK;
    }
    if (p.splits > 1) return launch_pipe_split(p, 1, weight, x, g, epi, no_fusion, (int)out_stride, num_output, partial, counters, stream);
#define LAUNCH_FC(BN_, GROUPS_)                                                                                                                                \
    hipLaunchKernelGGL((conv_nhwc_pipelined_kernel<64, BN_, PIPE_RING, false, 1, 1, GROUPS_>), grid, block, 0, stream, weight, x, g, epi, no_fusion, \
                       (int)out_stride, num_output, p.tiles_m, p.tiles_n, p.splits, p.steps_per_split, tile_magic(p.tiles_n), partial, counters, (const float*)0, 0, ConvShortcutArg<false>())
    if (p.bn == 256)
        LAUNCH_FC(256, 1);
    else if (p.bn == 128)
        LAUNCH_FC(128, 1);
    else if (p.groups == 4)
        LAUNCH_FC(64, 4);
    else
        LAUNCH_FC(64, 1);
#undef LAUNCH_FC
    return launch_status("conv_nhwc_pipelined_kernel<fc>");
}

// ---- InnerProduct through the K-split kernel on a scratch buffer the library holds itself, for callers that cannot
// allocate (under stream capture, in a serving loop that must not touch the allocator).  The array below is the
// workspace launch_fc_via_conv_pipelined otherwise gets from its caller; every device the library runs on holds its own
// copy of it, at its own address, until the process ends.
constexpr size_t STATIC_SCRATCH_PARTIAL_BYTES = 4u << 20;
constexpr size_t STATIC_SCRATCH_BYTES = SPLIT_COUNTER_BYTES + STATIC_SCRATCH_PARTIAL_BYTES;
static __device__ __align__(256) unsigned char scratch[STATIC_SCRATCH_BYTES];

constexpr int STATIC_SCRATCH_MAX_DEVICES = 64;
static void* g_scratch_ptr[STATIC_SCRATCH_MAX_DEVICES]; // device address of `scratch` on each device, 0 = not looked up yet
static std::mutex g_scratch_mutex;

// The array's name is only a handle on the host; its address on the CURRENT device comes from the runtime, once per device.
int static_scratch_for_current_device(void** ptr)
{
    int dev = 0;
    NCNNHIP_CHECK(hipGetDevice(&dev));
    NCNNHIP_REQUIRE(dev >= 0 && dev < STATIC_SCRATCH_MAX_DEVICES, "device %d beyond the %d the static scratch table covers", dev, STATIC_SCRATCH_MAX_DEVICES);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev])
    {
        void* p = 0;
        NCNNHIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        NCNNHIP_REQUIRE(p, "hipGetSymbolAddress returned a null address for the static scratch");
        g_scratch_ptr[dev] = p;
    }
    *ptr = g_scratch_ptr[dev];
    return NCNNHIP_OK;
}

// one workgroup: the arrival counters at the head of the scratch start every call at zero, whatever the last call left
__global__ __launch_bounds__(256) void clear_split_counters_kernel(unsigned* __restrict__ counters)
{
    for (int i = threadIdx.x; i < SPLIT_MAX_TILES; i += 256) counters[i] = 0u;
}

} // namespace ncnnhip

using namespace ncnnhip;

extern "C" int ncnnhip_innerproduct_int8_noalloc(const int8_t* x_dev, size_t x_stride, int rows, int num_input, int num_output, const int8_t* weight_dev,
                                                 const float* scale_in_dev, const float* bias_dev, ncnnhip_activation act, float* out_dev, size_t out_stride,
                                                 void* stream)
{
    NCNNHIP_REQUIRE(x_dev && weight_dev && scale_in_dev && out_dev, "ncnnhip_innerproduct_int8_noalloc: null pointer");
    NCNNHIP_REQUIRE(rows >= 1 && num_input >= 1 && num_output >= 1, "ncnnhip_innerproduct_int8_noalloc: bad shape");
    NCNNHIP_REQUIRE(x_stride >= (size_t)num_input && out_stride >= (size_t)num_output, "ncnnhip_innerproduct_int8_noalloc: stride too small");
    void* ptr = 0;
    int ret = static_scratch_for_current_device(&ptr);
    if (ret != NCNNHIP_OK) return ret;
    // few rows: the kernel that needs no scratch (and so no ordering between calls that share it)
    const bool aligned = ((reinterpret_cast<uintptr_t>(x_dev) | reinterpret_cast<uintptr_t>(weight_dev)) & 15) == 0 && x_stride % 16 == 0;
    if (aligned && fc_skinny_takes(rows, num_input, num_output))
        return ncnnhip_innerproduct_int8(x_dev, x_stride, rows, num_input, num_output, weight_dev, scale_in_dev, bias_dev, act, out_dev, out_stride, 0, stream);
    if (rows >= 8 && num_input % 64 == 0)
    {
        const size_t need = conv_nhwc_pipelined_workspace_words(num_output, rows, num_input / 64) * sizeof(int32_t);
        NCNNHIP_REQUIRE(need <= STATIC_SCRATCH_BYTES,
                        "ncnnhip_innerproduct_int8_noalloc: %d x %d -> %d needs %zu bytes of scratch, the library holds %zu; use ncnnhip_innerproduct_int8_ws",
                        rows, num_input, num_output, need, (size_t)STATIC_SCRATCH_BYTES);
        ConvEpilogue epi;
        epi.scale_in = scale_in_dev;
        epi.bias = bias_dev;
        epi.scale_out = 0;
        epi.act = act;
        epi.out = out_dev;
        epi.out_cstep = epi.out_nstep = 0;
        epi.pix_per_img = rows;
        epi.batch = 1;
        epi.out_channel0 = 0;
        epi.num_output = num_output;
        epi.acc_out = 0;
        if (need)
        {
            hipLaunchKernelGGL(clear_split_counters_kernel, dim3(1), dim3(256), 0, as_stream(stream), (unsigned*)ptr);
            ret = launch_status("clear_split_counters_kernel");
            if (ret != NCNNHIP_OK) return ret;
        }
        bool handled = false;
        ret = launch_fc_via_conv_pipelined(x_dev, x_stride, rows, num_input, num_output, weight_dev, epi, out_stride, ptr, STATIC_SCRATCH_BYTES,
                                           as_stream(stream), &handled);
        if (handled) return ret;
    }
    // shapes the matrix-core kernel does not take run on the kernel that needs no scratch at all
    return ncnnhip_innerproduct_int8(x_dev, x_stride, rows, num_input, num_output, weight_dev, scale_in_dev, bias_dev, act, out_dev, out_stride, 0, stream);
}
