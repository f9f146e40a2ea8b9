// The launch plans of the kernels, which are plain host arithmetic, for the tests (host_plans.py).
#include <chrono>

#include "gs2d_direct_plan.hpp"
#include "gs2d_grad_grid_plan.hpp"
#include "gs_grad_gather_plan.hpp"
#include "gs_grad_tiles_plan.hpp"
#include "resize_flat_plan.hpp"
#include "resize_grad_plan.hpp"
#include "resize_nearest_plan.hpp"
#include "resize_nhwc_plan.hpp"

using namespace opscv;

extern "C" {

// tiles, channel runs; 0 where the tiled kernel is not taken
int direct_tiles(int elem, int64_t N, int64_t C, int64_t Hin, int64_t Win, int64_t Hout, int64_t Wout, int64_t* out)
{
    GridSamplerArgs a;
    a.elem = (Elem)elem;
    a.N = N;
    a.C = C;
    a.Hin = Hin;
    a.Win = Win;
    a.Hout = Hout;
    a.Wout = Wout;
    const DirectTilePlan p = direct_tile_plan(a);
    out[0] = p.tiles;
    out[1] = p.chan_runs;
    return p.ok ? 1 : 0;
}

// tile rows, workgroups, planes a workgroup walks at most; 0 where the planes kernel is not taken.  Gradient of (Hs, Ws)
// from (Hd, Wd), dense planes on a 16-byte boundary.
static ResizeGradArgs resize_grad_args(int elem, int64_t planes, int64_t Hs, int64_t Ws, int64_t Hd, int64_t Wd, int align)
{
    ResizeGradArgs a;
    a.elem_in = a.elem_out = (Elem)elem;
    a.half_pixel = align ? 0 : 1;
    a.N = 1;
    a.C = planes;
    a.Hs = Hs;
    a.Ws = Ws;
    a.Hd = Hd;
    a.Wd = Wd;
    auto scale = [&](int64_t s, int64_t d) {
        return align ? (d > 1 ? (float)(s - 1) / (float)(d - 1) : 0.0f) : (float)s / (float)d;
    };
    a.scale_h = scale(Hs, Hd);
    a.scale_w = scale(Ws, Wd);
    return a;
}

int resize_grad_planes(int elem, int64_t planes, int64_t Hs, int64_t Ws, int64_t Hd, int64_t Wd, int align, int64_t* out)
{
    const PlaneTile t = plane_tile(resize_grad_args(elem, planes, Hs, Ws, Hd, Wd, align));
    out[0] = t.rows;
    out[1] = t.blocks;
    out[2] = (planes + t.slots - 1) / (t.slots > 0 ? t.slots : 1);
    return t.rows > 0 ? 1 : 0;
}

// rows of a wavefront, whether a lane moves two units of a row, rows an element may visit; 0 where the
// rows kernel is not taken
int resize_grad_rows(int elem, int64_t planes, int64_t Hs, int64_t Ws, int64_t Hd, int64_t Wd, int align, int64_t* out)
{
    const RowsPlan p = rows_plan(resize_grad_args(elem, planes, Hs, Ws, Hd, Wd, align));
    out[0] = p.rows;
    out[1] = p.two ? 1 : 0;
    out[2] = p.visits;
    return p.ok ? 1 : 0;
}

// kernel of a call: 1 rows, 2 planes, 3 LDS tiles, 4 gather
int resize_grad_kernel(int elem, int64_t planes, int64_t Hs, int64_t Ws, int64_t Hd, int64_t Wd, int align, int64_t* out)
{
    out[0] = (int64_t)resize_grad_plan(resize_grad_args(elem, planes, Hs, Ws, Hd, Wd, align)).kernel;
    return 1;
}

// most rows, and columns, an outgoing element may visit in the rows kernel
int resize_grad_rows_visits(int64_t* out)
{
    out[0] = kRowsColumns;
    return 1;
}

// estimates of the input gradient of planes (nanoseconds): elections, sorting; 0 where the elections run
int sorting_takes_planes(int elem, int64_t interp, int64_t N, int64_t C, int64_t H, int64_t W, int64_t points, int64_t* out)
{
    GradGatherArgs a;
    a.elem = (Elem)elem;
    a.interp = (int)interp;
    a.N = N;
    a.C = C;
    a.H = H;
    a.W = W;
    a.points = points;
    const PlaneGradTimes t = plane_grad_times(a);
    out[0] = (int64_t)(t.elections * 1e3);
    out[1] = (int64_t)(t.sorting * 1e3);
    return sorting_takes_planes(a) && gather_plan(a).ok ? 1 : 0;
}

// 1: channels-last rows that shrink from Hs to Hd go in pairs
int shrink_in_pairs(int64_t unit, int64_t Hs, int64_t Hd, int align)
{
    ResizeArgs a;
    a.half_pixel = align ? 0 : 1;
    a.scale_h = align ? (float)(Hs - 1) / (float)(Hd - 1) : (float)Hs / (float)Hd;
    return shrinking_rows_go_in_pairs(a, (int)unit) ? 1 : 0;
}

// flat resize: non-temporal stores, rows of a group in runs
int flat_resize(int elem, int64_t planes, int64_t Hs, int64_t Ws, int64_t Hd, int64_t Wd, int64_t* out)
{
    ResizeArgs a;
    a.elem = (Elem)elem;
    a.N = 1;
    a.C = planes;
    a.Hs = Hs;
    a.Ws = Ws;
    a.Hd = Hd;
    a.Wd = Wd;
    const FlatStores s = flat_stores(a);
    out[0] = s.streaming;
    out[1] = s.runs;
    return 1;
}

// sorting variant of the input gradient: items run at a time, 32-bit words of an item; 0 where it cannot run
int gather_groups(int elem, int64_t interp, int64_t N, int64_t C, int64_t D, int64_t H, int64_t W, int64_t points, int64_t* out)
{
    GradGatherArgs a;
    a.elem = (Elem)elem;
    a.dim = D > 0 ? 3 : 2;
    a.interp = (int)interp;
    a.N = N;
    a.C = C;
    a.D = D > 0 ? D : 1;
    a.H = H;
    a.W = W;
    a.points = points;
    const GatherPlan p = gather_plan(a);
    out[0] = p.group;
    out[1] = p.p.lay.item_words;
    return p.ok ? 1 : 0;
}

// input gradient by tiles: items run at a time, 32-bit words of an item, tiles, blocks of points, channel blocks; 0 where the
// lists of gather_groups take it
int gradient_tiles(int elem, int64_t interp, int64_t pad, int64_t N, int64_t C, int64_t D, int64_t H, int64_t W, int64_t points,
                   int64_t per_core, int64_t* out)
{
    GradGatherArgs a;
    a.elem = (Elem)elem;
    a.dim = D > 0 ? 3 : 2;
    a.interp = (int)interp;
    a.pad = (int)pad;
    a.N = N;
    a.C = C;
    a.D = D > 0 ? D : 1;
    a.H = H;
    a.W = W;
    a.points = points;
    a.items_per_core = per_core;
    const TilesPlan p = tiles_plan(a);
    out[0] = p.group;
    out[1] = p.p.lay.item_words;
    out[2] = p.p.tiles;
    out[3] = p.p.blocks;
    out[4] = p.cblocks;
    return p.ok ? 1 : 0;
}

// the grid gradient's tiles: tiles, workgroups; 0 where its points are taken in rows
int grid_gradient_tiles(int elem, int64_t interp, int64_t N, int64_t H, int64_t W, int64_t Ho, int64_t Wo, int64_t* out)
{
    GridSamplerGradArgs a;
    a.elem = (Elem)elem;
    a.interp = (int)interp;
    a.N = N;
    a.C = 1;
    a.Hin = H;
    a.Win = W;
    a.Hout = Ho;
    a.Wout = Wo;
    const GridTilePlan p = grid_tile_plan(a);
    out[0] = p.tiles;
    out[1] = p.blocks;
    return p.ok ? 1 : 0;
}

// points and contributions of an element beyond which a tile is the crowded tiles' kernel's
int crowded_tiles(int elem, int64_t interp, int64_t pad, int64_t N, int64_t C, int64_t dim, int64_t* out)
{
    GradGatherArgs a;
    a.elem = (Elem)elem;
    a.dim = (int)dim;
    a.interp = (int)interp;
    a.pad = (int)pad;
    a.N = N;
    a.C = C;
    const CrowdedTile t = crowded_tile(a);
    out[0] = t.points;
    out[1] = t.contributions;
    return 1;
}

// nearest resize by runs of rows: rows of a run, pieces of a row, elements of a piece, bytes of LDS; 0 where another kernel
// takes it.  `in_chunks`: source rows on the 16-byte grid
int nearest_rows(int elem, int64_t N, int64_t C, int64_t Hs, int64_t Ws, int64_t Hd, int64_t Wd, int64_t last, int64_t in_chunks,
                 int64_t* out)
{
    ResizeArgs a;
    a.elem = (Elem)elem;
    a.mode = ResizeMode::Nearest;
    a.channels_last = (int)last;
    a.N = N;
    a.C = C;
    a.Hs = Hs;
    a.Ws = Ws;
    a.Hd = Hd;
    a.Wd = Wd;
    a.scale_h = (float)Hs / (float)Hd;
    a.scale_w = (float)Ws / (float)Wd;
    const NearestRows p = nearest_rows_plan(a, in_chunks != 0);
    out[0] = p.run;
    out[1] = p.chunks;
    out[2] = p.cols;
    out[3] = p.lds_bytes;
    return p.run > 0 ? 1 : 0;
}

// nanoseconds that nearest_rows takes, the least of twenty runs of 50
int64_t nearest_rows_nanoseconds(int elem, int64_t N, int64_t C, int64_t Hs, int64_t Ws, int64_t Hd, int64_t Wd, int64_t last)
{
    int64_t least = INT64_MAX, out[4];
    for (int run = 0; run < 20; run++) {
        const auto start = std::chrono::steady_clock::now();
        for (int i = 0; i < 50; i++) {
            nearest_rows(elem, N, C, Hs, Ws, Hd, Wd, last, 0, out);
        }
        const int64_t t = std::chrono::duration_cast<std::chrono::nanoseconds>(std::chrono::steady_clock::now() - start).count() / 50;
        least = t < least ? t : least;
    }
    return least;
}

}  // extern "C"
