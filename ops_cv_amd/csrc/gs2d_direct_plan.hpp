// Launch plan of the direct sampler's tiled kernel (gs2d_kernels.hip): host arithmetic only.
#pragma once

#include <cstdint>

#include "acl_types.hpp"
#include "launch_limits.hpp"

namespace opscv {

constexpr int kDirectThreads = 256;
constexpr int kPatchW = 16, kPatchH = 4, kPatches = 2;
constexpr int kTileCols = 2 * kPatchW, kTileLines = 2 * kPatches * kPatchH;
static_assert(kTileCols * kTileLines == kPatches * kDirectThreads, "four wavefronts, two by two");

struct DirectTilePlan {
    bool ok = false;
    int64_t tiles_x = 0, tiles_y = 0, tiles = 0;
    int64_t chan_run = 0, chan_runs = 0;  // channels of a workgroup, and how many such runs there are
};

// A workgroup per CU.  Below, a wavefront's two patches are a chain twice as long as a lane's one pixel, and for bicubic
// samples more: fp32 1x3x300x300 -> 16x32 bilinear 3.4 us in the row order, 4.3 in tiles, bicubic 4.5 / 11.  Tiles against
// row order over 1200 launches, medians: under 64 workgroups bilinear 1.08, nearest 1.01, bicubic 1.65, 64 to 256 1.05,
// 1.05 and 1.10, 256 to 512 0.99 to 1.01, from 1024 on 0.75 to 0.99.
constexpr int64_t kTileFewest = 256;

// Tiles where lines are shared between the rows of an output: planes beyond the 32 KiB of a CU's first-level cache.
// Counts that fit the launch, offsets in a plane that fit 32 bits; anything larger goes to the kernel that walks its
// pixels with as many workgroups as it likes.
inline DirectTilePlan direct_tile_plan(const GridSamplerArgs& a)
{
    DirectTilePlan p;
    const int64_t esz = elem_size(a.elem);
    const int64_t limit = INT32_MAX / esz;
    p.tiles_x = (a.Wout + kTileCols - 1) / kTileCols;
    p.tiles_y = (a.Hout + kTileLines - 1) / kTileLines;
    if (a.Win < 2 || a.Hin * a.Win * esz <= (32 << 10) || a.Hin * a.Win > limit || a.Wout < kTileCols ||
        a.Hout < kTileLines || a.Hout > limit / a.Wout || a.N > (int64_t)UINT32_MAX / (p.tiles_x * p.tiles_y) ||
        !fits_launch(a.N * p.tiles_x * p.tiles_y, kDirectThreads)) {
        return p;
    }
    p.tiles = a.N * p.tiles_x * p.tiles_y;
    // runs of channels to different workgroups where the tiles alone are too few, as in run_direct
    int64_t chunks = (4096 + p.tiles - 1) / p.tiles;
    chunks = chunks < a.C ? chunks : a.C;
    p.chan_run = (a.C + chunks - 1) / chunks;
    p.chan_run = (p.chan_run + 3) / 4 * 4;
    p.chan_runs = (a.C + p.chan_run - 1) / p.chan_run;
    p.ok = p.chan_runs <= 65535 && p.tiles * p.chan_runs >= kTileFewest;
    return p;
}

}  // namespace opscv
