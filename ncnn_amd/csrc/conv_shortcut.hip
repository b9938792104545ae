// A residual block's two 1x1 convolutions into one sum, where the block has a projection shortcut: the pipelined kernel with the shortcut's
// K steps in front of the main convolution's (MODE 4), for layers with many tiles; conv_stream.hip has the form for few.
//
// The shortcut's fp32 result is neither written nor read again: for ResNet-50's second stage at 16 images 51 MB each way, half of
// the traffic of the two launches, which moved it at 5.5 TB/s.  The one launch is not at that rate (128 images 3.7 TB/s there, 1.3 in the last stage):
// one to eight K steps of each convolution, two epilogues and the stores follow one another with nothing of the next tile under way.
#include "conv_nhwc_pipelined_kernel.h"

namespace ncnnhip {

// Here a workgroup walks both K whole behind one barrier a step, where each convolution alone would share its K between sixteen wavefronts or split it over
// workgroups (up to 256 tiles) or run on wider tiles (many): what the launch saves is a launch and the fp32 blob, what it loses grows with the steps (64 of K).
// Time of one launch over that of two, fp32 and quantised output (main + shortcut steps; tiles of 64 x 64):
//   160 tiles   1 + 1 0.70, 4 + 8 0.87, 6 + 12 0.95, 8 + 16 1.09, 16 + 32 1.37; 1 + 16 0.98, 11 + 1 0.94
//   400         1 + 1 0.68, 8 + 16 0.95, 10 + 20 1.00, 12 + 24 1.04, 16 + 32 1.08
//   784         1 + 1 0.66, 8 + 16 0.94, 12 + 24 1.01, 16 + 32 1.07
//   3136        1 + 1 0.60, 4 + 8 0.81, 8 + 16 0.99, 10 + 20 1.08, 12 + 24 1.11
bool conv_shortcut_pays(const NhwcGeom& g, int shortcut_steps)
{
    if (conv_stream_shortcut_tile(g, shortcut_steps)) return true;
    const int steps = g.K / 64;
    const long long tiles = (long long)ceil_div(g.npix, 64) * ceil_div(g.cout, 64);
    if (tiles <= 256) return steps <= 12 && steps + shortcut_steps <= 18;
    return steps + shortcut_steps <= (tiles <= 512 ? 30 : tiles <= 2048 ? 36 : 24);
}

int launch_conv_shortcut(const NhwcGeom& g_in, const int8_t* wpk, const int8_t* x, const ConvShortcut& sc, const ConvEpilogue& epi, const ConvFusion& fusion, int out_cp,
                         hipStream_t stream)
{
    const long long sc_bytes = (long long)(g_in.npix / (sc.outw * sc.outh)) * sc.H * sc.W * sc.Cp;
    if (conv_stream_shortcut_tile(g_in, sc.Cp / 64) && sc_bytes < (1ll << 31)) return launch_conv_stream_shortcut(g_in, wpk, x, sc, epi, fusion, out_cp, stream);
    NhwcGeom g = g_in;
    g.H = g.outh = 1;
    g.W = g.outw = g.npix;
    // K stays whole: the shortcut's sums are finished where the main ones are.  64-channel tiles (five workgroups to a unit where three of 128 channels
    // fit) until there are so many that the activations read per tile weigh more.  us, 128 channels wide / 64, fp32 and quantised output:
    // 16 images 64 + 64 -> 256 on 56 x 56 22.2 / 18.8, 128 + 256 -> 512 on 28 x 28 19.5 / 15.7, 256 + 512 -> 1024 on 14 x 14 14.5 / 13.4, 512 + 1024 -> 2048
    // on 7 x 7 18.5 / 14.6 (two launches 36.5, 26.6, 17.4, 15.9); 64 images 80 / 84 (12544 tiles; int8 alone 57 / 50), 44.9 / 44.4 (6272), 37.1 / 34.4, 37.8 / 32.1; 128 images 128 + 256 -> 512
    // (12544 tiles of six steps) 93.2 / 86.4.
    const int tiles_m = ceil_div(g.npix, 64);
    const long long narrow = (long long)tiles_m * ceil_div(g.cout, 64);
    const bool wide = !tiles_fit_a_launch(tiles_m, ceil_div(g.cout, 64)) || (narrow >= 8192 && g.K / 64 + sc.Cp / 64 <= 4);
    const int tiles_n = ceil_div(g.cout, wide ? 128 : 64);
    const long long blocks = (long long)tiles_m * tiles_n;
    NCNNHIP_REQUIRE(tiles_fit_a_launch(tiles_m, tiles_n), "convolution: too many tiles");
    ConvShortcutArg<true> arg;
    static_cast<ConvShortcut&>(arg) = sc;
#define LAUNCH_SHORTCUT(BN_)                                                                                                                            \
    hipLaunchKernelGGL((conv_nhwc_pipelined_kernel<64, BN_, PIPE_RING, false, 4>), dim3((unsigned)blocks), dim3(256), 0, stream, wpk, x, g, epi, fusion, out_cp, out_cp, \
                       tiles_m, tiles_n, 1, g.K / 64, tile_magic(tiles_n), (int32_t*)0, (unsigned*)0, (const float*)0, 0, arg)
    if (wide)
        LAUNCH_SHORTCUT(128);
    else
        LAUNCH_SHORTCUT(64);
#undef LAUNCH_SHORTCUT
    return launch_status("conv_nhwc_pipelined_kernel (shortcut)");
}

} // namespace ncnnhip
