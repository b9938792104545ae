// Launches of the pipelined channels-last convolution kernel with K split over workgroups (few output tiles, long K:
// the partial sums meet in a workspace, the last workgroup of a tile to finish runs the epilogue).  The kernel itself is in conv_nhwc_pipelined_kernel.h.
// Tiles of 64 x 64 alone: the planner splits K below 256 tiles, and there it has made them that small.
#include "conv_nhwc_pipelined_kernel.h"

namespace ncnnhip {

int launch_pipe_split(const PipePlan& p, int mode, const int8_t* wpk, const int8_t* x, const NhwcGeom& g, const ConvEpilogue& epi, const ConvFusion& fusion,
                      int out_cp, int col_limit, int32_t* partial, unsigned* counters, hipStream_t stream)
{
    NCNNHIP_REQUIRE(p.splits > 1 && partial && counters && (mode == 0 || mode == 1 || mode == 3), "convolution: K split without its workspace");
    NCNNHIP_REQUIRE(p.bm == 64 && p.bn == 64, "convolution: K split of %d x %d tiles", p.bm, p.bn);
    dim3 grid((unsigned)((long long)p.tiles_m * p.tiles_n * p.splits)), block((unsigned)(256 * p.groups));
#define LAUNCH_SPLIT(MODE_, GROUPS_)                                                                                                                             \
    hipLaunchKernelGGL((conv_nhwc_pipelined_kernel<64, 64, PIPE_RING, true, MODE_, 1, GROUPS_>), grid, block, 0, stream, wpk, x, g, epi, fusion, out_cp, col_limit, \
                       p.tiles_m, p.tiles_n, p.splits, p.steps_per_split, tile_magic(p.tiles_n), partial, counters, (const float*)0, 0, ConvShortcutArg<false>())
#define LAUNCH_SPLIT_MODE(GROUPS_)   \
    do                               \
    {                                \
        if (mode == 1)               \
            LAUNCH_SPLIT(1, GROUPS_); \
        else if (mode == 3)          \
            LAUNCH_SPLIT(3, GROUPS_); \
        else                         \
            LAUNCH_SPLIT(0, GROUPS_); \
    } while (0)
    if (p.groups == 4)
        LAUNCH_SPLIT_MODE(4);
    else
        LAUNCH_SPLIT_MODE(1);
#undef LAUNCH_SPLIT_MODE
#undef LAUNCH_SPLIT
    return launch_status("conv_nhwc_pipelined_kernel (K split)");
}

} // namespace ncnnhip
