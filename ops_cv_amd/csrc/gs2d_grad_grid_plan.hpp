// Launch plan of the grid gradient's tiles (gs2d_grad.hip): host arithmetic only.
#pragma once

#include <cstdint>

#include "acl_types.hpp"
#include "gs_grad_gather_plan.hpp"
#include "launch_limits.hpp"

namespace opscv {

constexpr int kGridTile = 16;  // square: a lane per grid point of 256
constexpr int kGridTileThreads = kGridTile * kGridTile;

// Few points are bound by the lines that a CU's loads touch, one wavefront's channel after the other: workgroups of a wavefront
// bring them to four times as many CUs, neighbours on one XCD (in turn over all of them every XCD's L2 fetches most of the planes:
// fp32 1x155x72x88 -> 69x84 17.4 us with 256 threads, 20.7 in turn, 16.8 so, fp16 16x111x27x50 -> 18x33 16.9 / 18.3 / 14.5, fp32
// 12x68x44x46 12.4 / 12.4 / 9.0).  256 / 64 threads, grid gradient alone: bicubic fp32 10x54x32x24 -> 62x46 (28520 points) 47.8 / 41.0
// us, 2x256x56x80 -> 101x145 at random 359 / 208, bilinear bf16 8x52x32x32 -> 61x61 9.9 / 8.5, fp32 1x79x133x238 at random 42.3 / 25.4;
// 130 draws 1.17 and 1.29 times as fast, four of them slower, one large plane after the other in smooth grids: bicubic fp32 1x200x152x184
// 181 / 193, fp16 1x201x72x88 -> 112x136 102 / 110.  Beyond, with more wavefronts than two a CU, it depends (measured in turn over
// the XCDs): 27x51x32x48 (41472 points) 9.9 / 10.8, bicubic 21x5x85x85 -> 45x45 (42525) 12.4 / 11.2, 24x49x42x79 (79632) 15.5 / 19.8.
// (A wavefront for either sum of 64 points instead: 47.6 / 48.4 on the first.)
constexpr int64_t kGridSpreadPoints = 32768;
constexpr int kGridSpreadThreads = 64;

struct GridTilePlan {
    bool ok = false;
    int64_t tiles_x = 0, per_item = 0, tiles = 0;
    int64_t blocks = 0;  // as many for every XCD
};

// Tiles of grid points for the grid gradient: planes beyond the first-level cache, where lines are fetched again for every
// row of points, two workgroups per CU, and few lanes along the edges without a point.  Rows / tiles, both gradients' grid
// part alone: fp32 8x3x479x637 40.5 / 33.2 us, fp16 6x3x576x472 -> 362x297 15.8 / 11.3, fp32 2x37x132x184 11.7 / 9.6; smaller
// planes bf16 2x105x90x146 19.4 / 24.4, fp16 19x11x144x120 -> 210x175 22.6 / 23.8; few tiles fp32 3x3x241x369 -> 128x196 7.0 /
// 7.2.
//
// Not for bicubic samples, whose sixteen taps share lines within a point already: fp32 8x3x479x637 115 / 138 us, fp16 108 / 153,
// fp32 2x3x720x1280 106 / 120, 1x4x256x256 -> 512x512 18.0 / 23.5, with border padding 19.6 / 32.3, 4x1x300x400 17.2 / 19.4.
inline GridTilePlan grid_tile_plan(Elem elem, int interp, int64_t N, int64_t H, int64_t W, int64_t Ho, int64_t Wo)
{
    GridTilePlan p;
    if (interp != 0 || N < 1 || Ho < 1 || Wo < 1 || Ho > INT32_MAX / 2 || Wo > INT32_MAX / 2 || N > INT32_MAX / 2) {
        return p;
    }
    const int64_t tiles_y = (Ho + kGridTile - 1) / kGridTile;
    p.tiles_x = (Wo + kGridTile - 1) / kGridTile;
    p.per_item = p.tiles_x * tiles_y;
    if (p.per_item > INT32_MAX / 2 / N) {
        return p;
    }
    p.tiles = N * p.per_item;
    p.blocks = (p.tiles + 7) / 8 * 8;
    const int64_t lanes = p.per_item * kGridTileThreads;
    p.ok = H * W * elem_size(elem) > (64 << 10) && p.tiles >= 512 && lanes - lanes / 5 <= Ho * Wo &&
           fits_launch(p.blocks, kGridTileThreads);
    return p;
}

inline GridTilePlan grid_tile_plan(const GridSamplerGradArgs& a)
{
    return grid_tile_plan(a.elem, a.interp, a.N, a.Hin, a.Win, a.Hout, a.Wout);
}

inline GridTilePlan grid_tile_plan(const GradGatherArgs& a)
{
    return grid_tile_plan(a.elem, a.interp, a.N, a.H, a.W, a.Ho, a.Wo);
}

}  // namespace opscv
