// Launches of the pipelined channels-last convolution kernel with K split over workgroups (few output tiles, long K:
// the partial sums meet in a workspace, the last workgroup of a tile to finish runs the epilogue).  The kernel itself is in conv_nhwc_pipelined_kernel.h.
#include "conv_nhwc_pipelined_kernel.h"

namespace ncnnhip {

int launch_pipe_split(const PipePlan& p, int mode, const int8_t* wpk, const int8_t* x, const NhwcGeom& g, const ConvEpilogue& epi, const ConvFusion& fusion,
                      int out_cp, int col_limit, int32_t* partial, unsigned* counters, hipStream_t stream)
{
    NCNNHIP_REQUIRE(p.splits > 1 && partial && counters && (mode == 0 || mode == 1 || mode == 3), "convolution: K split without its workspace");
    dim3 grid((unsigned)((long long)p.tiles_m * p.tiles_n * p.splits)), block((unsigned)(256 * p.groups));
#define LAUNCH_SPLIT_MODE(BM_, BN_, MODE_, GROUPS_)                                                                                                              \
    hipLaunchKernelGGL((conv_nhwc_pipelined_kernel<BM_, BN_, PIPE_RING, true, MODE_, 1, GROUPS_>), grid, block, 0, stream, wpk, x, g, epi, fusion, out_cp, \
                       col_limit, p.tiles_m, p.tiles_n, p.splits, p.steps_per_split, tile_magic(p.tiles_n), partial, counters, (const float*)0, 0, ConvShortcutArg<false>())
#define LAUNCH_SPLIT(BM_, BN_, GROUPS_)         \
    do                                          \
    {                                           \
        if (mode == 1)                          \
            LAUNCH_SPLIT_MODE(BM_, BN_, 1, GROUPS_);     \
        else if (mode == 3)                     \
            LAUNCH_SPLIT_MODE(BM_, BN_, 3, GROUPS_);     \
        else                                    \
            LAUNCH_SPLIT_MODE(BM_, BN_, 0, GROUPS_);     \
    } while (0)
    if (p.bm == 128 && p.bn == 256)
        LAUNCH_SPLIT(128, 256, 1);
    else if (p.bm == 128 && p.bn == 128)
        LAUNCH_SPLIT(128, 128, 1);
    else if (p.bm == 128)
        LAUNCH_SPLIT(128, 64, 1);
    else if (p.bn == 256)
        LAUNCH_SPLIT(64, 256, 1);
    else if (p.bn == 128)
        LAUNCH_SPLIT(64, 128, 1);
    else if (p.groups == 4)
        LAUNCH_SPLIT(64, 64, 4);
    else
        LAUNCH_SPLIT(64, 64, 1);
#undef LAUNCH_SPLIT
#undef LAUNCH_SPLIT_MODE
    return launch_status("conv_nhwc_pipelined_kernel (K split)");
}

} // namespace ncnnhip
