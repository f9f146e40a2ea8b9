// The samplers' gradient of the grid by a lane per grid point: for a kernel of its own (gs2d_grad.hip, gs3d_grad.hip) and for the
// first kernel of the input gradient by tiles, which has room beside it (gs_grad_tiles.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "fast_div.hpp"
#include "gs2d_grad_grid_plan.hpp"
#include "gs2d_grad_math.hpp"
#include "gs3d_grad_math.hpp"
#include "gs_grad_gather_plan.hpp"

namespace opscv {

struct Grid2Params {
    int32_t C, H, W, Ho, Wo;
    int32_t pad, align;
    int32_t blocks_per_item;  // points in rows: see gs2d_grid_gradient_block
    uint32_t pieces;          // in tiles: how many, and how they are numbered; in rows: workgroups dealt out by XCD, 0: in turn
    FastDiv by_item, by_tiles_x;
    int64_t total;            // points of the batch
};

struct Grid2Launch {
    bool ok = false, tiled = false;
    Grid2Params p{};
    int64_t blocks = 0;  // of as many threads as grid2_launch was asked for
};

inline Grid2Launch grid2_launch(const GradGatherArgs& a, int threads = kGridTileThreads)
{
    Grid2Launch g;
    g.p.C = (int32_t)a.C;
    g.p.H = (int32_t)a.H;
    g.p.W = (int32_t)a.W;
    g.p.Ho = (int32_t)a.Ho;
    g.p.Wo = (int32_t)a.Wo;
    g.p.pad = a.pad;
    g.p.align = a.align;
    g.p.total = a.N * a.points;
    if (const GridTilePlan t = grid_tile_plan(a); t.ok) {
        g.tiled = true;
        g.p.pieces = (uint32_t)t.tiles;
        g.p.by_item = make_fast_div((uint32_t)t.per_item);
        g.p.by_tiles_x = make_fast_div((uint32_t)t.tiles_x);
        g.blocks = t.blocks;
    } else {
        g.blocks = (g.p.total + threads - 1) / threads;
        const int64_t per_item = a.points / threads;
        g.p.blocks_per_item = (a.points % threads == 0 && a.N % 8 == 0 && per_item <= INT32_MAX) ? (int32_t)per_item : 0;
        if (threads == kGridSpreadThreads && g.p.blocks_per_item == 0 && g.blocks <= INT32_MAX - 8) {
            g.p.pieces = (uint32_t)g.blocks;
            g.blocks = (g.blocks + 7) / 8 * 8;
        }
    }
    g.ok = g.blocks <= INT32_MAX;
    return g;
}

// One lane per grid point.  TILED: a workgroup takes 16 x 16 points of an item, a wavefront 16 x 4 of them, so that under a
// turned grid the corners of its points share cache lines in both directions: 64 points of a row lie in up to 64 lines of a
// plane.  XCD k takes the k-th eighth of the workgroups, so that neighbouring tiles share an L2.
//
// Bound by the lines that the gathers touch and their latency: the loads of up to eight channels are on their way together,
// of fewer channels all of them (fp32 8x3x479x637, rotations of up to 30 degrees: 58 us in rows, a channel after the other;
// 40 with the three channels' loads together; 33 in tiles).  Bicubic samples have the sixteen loads of a channel on their way
// together, in rows (grid_tile_plan): turned grids, one load after the other / together, fp32 8x3x479x637 114 / 115 us, 2x64x128x128
// 72 / 62, 8x128x32x32 114 / 116, fp16 134 / 108, 156 / 62, 190 / 101; points at random, whose lines are seldom in the cache, fp32
// 393 / 395, 118 / 125, 108 / 117, fp16 373 / 370, 154 / 107, 188 / 115.
template <typename T, int INTERP, bool TILED, int THREADS = kGridTileThreads>
__device__ __forceinline__ void gs2d_grid_gradient_block(uint32_t block_index, const T* __restrict__ gout, const T* __restrict__ x,
                                                         const T* __restrict__ grid, T* __restrict__ dgrid, const Grid2Params& p)
{
    using Taps = GradTaps<T, INTERP>;
    const int32_t points = p.Ho * p.Wo;
    int64_t n, idx;
    int32_t pt;
    if constexpr (TILED) {
        const uint32_t per_xcd = p.pieces / 8u + (p.pieces % 8u != 0u ? 1u : 0u);
        const uint32_t piece = (block_index & 7u) * per_xcd + (block_index >> 3);
        if ((block_index >> 3) >= per_xcd || piece >= p.pieces) {
            return;
        }
        const uint32_t item = fast_div(piece, p.by_item), tile = piece - item * p.by_item.div;
        const uint32_t ty = fast_div(tile, p.by_tiles_x), tx = tile - ty * p.by_tiles_x.div;
        const int32_t px = (int32_t)(tx * kGridTile + threadIdx.x % kGridTile);
        const int32_t py = (int32_t)(ty * kGridTile + threadIdx.x / kGridTile);
        if (px >= p.Wo || py >= p.Ho) {
            return;
        }
        n = item;
        pt = py * p.Wo + px;
        idx = n * points + pt;
    } else {
        // blocks_per_item > 0: workgroups are handed to the 8 XCDs round-robin by index; all workgroups of one batch item
        // go to one XCD, so that the planes of that item (every lane walks all of them) are fetched into one L2 once
        // instead of into all eight (fp16 N16 C256 64x64: 185.6 MB fetched for 67.1 MB of operands otherwise).  The launch
        // plan asks for it when the items divide evenly among the XCDs and the workgroups evenly among the items.
        uint32_t block = block_index;
        if (p.blocks_per_item > 0) {
            const uint32_t xcd = block_index & 7u, i = block_index >> 3;
            block = ((i / (uint32_t)p.blocks_per_item) * 8u + xcd) * (uint32_t)p.blocks_per_item + i % (uint32_t)p.blocks_per_item;
        } else if (p.pieces > 0) {  // XCD k takes the k-th eighth of the workgroups, as in tiles
            block = (block_index & 7u) * ((p.pieces + 7u) / 8u) + (block_index >> 3);
            if (block >= p.pieces) {
                return;
            }
        }
        idx = (int64_t)block * THREADS + threadIdx.x;
        if (idx >= p.total) {
            return;
        }
        n = idx / points;
        pt = (int32_t)(idx - n * points);
    }
    if (INTERP == 1) {
        ElemIO<T>::store(dgrid + 2 * idx, 0.0f);
        ElemIO<T>::store(dgrid + 2 * idx + 1, 0.0f);
        return;
    }
    Taps tp;
    decide_grad_taps<T, INTERP>(tp, ElemIO<T>::load(grid + 2 * idx), ElemIO<T>::load(grid + 2 * idx + 1), p.H, p.W,
                                p.pad, p.align);
    const int32_t plane_px = p.H * p.W;
    const T* x_n = x + n * p.C * (int64_t)plane_px;
    const T* go_n = gout + n * p.C * (int64_t)points + pt;
    float gix = 0.0f, giy = 0.0f;
    // f(number of channels, first channel): the sums run over the channels in order; the loads do not depend on them, so
    // they are issued a group of channels ahead (a lane has one grid point and would otherwise wait out every load in turn)
    auto for_groups = [&](auto&& f) __attribute__((always_inline)) {
        int32_t c = 0;
        for (; c + 8 <= p.C; c += 8) {
            f(std::integral_constant<int, 8>{}, c);
        }
        if (c + 4 <= p.C) {
            f(std::integral_constant<int, 4>{}, c);
            c += 4;
        }
        switch (p.C - c) {
            case 3: f(std::integral_constant<int, 3>{}, c); break;
            case 2: f(std::integral_constant<int, 2>{}, c); break;
            case 1: f(std::integral_constant<int, 1>{}, c); break;
            default: break;
        }
    };
    if (INTERP == 0) {
        const float dxe = (float)(tp.x0 == INT32_MAX ? tp.x0 : tp.x0 + 1) - tp.fx, dxw = tp.fx - (float)tp.x0;
        const float dys = (float)(tp.y0 == INT32_MAX ? tp.y0 : tp.y0 + 1) - tp.fy, dyn = tp.fy - (float)tp.y0;
        const bool ok0 = tp.off[0] >= 0, ok1 = tp.off[1] >= 0, ok2 = tp.off[2] >= 0, ok3 = tp.off[3] >= 0;
        const int32_t o0 = ok0 ? tp.off[0] : 0, o1 = ok1 ? tp.off[1] : 0, o2 = ok2 ? tp.off[2] : 0,
                      o3 = ok3 ? tp.off[3] : 0;
        auto accumulate = [&](float go, float v0, float v1, float v2, float v3) __attribute__((always_inline)) {
            if (ok0) {
                gix -= v0 * dys * go;
                giy -= v0 * dxe * go;
            }
            if (ok1) {
                gix += v1 * dys * go;
                giy -= v1 * dxw * go;
            }
            if (ok2) {
                gix -= v2 * dyn * go;
                giy += v2 * dxe * go;
            }
            if (ok3) {
                gix += v3 * dyn * go;
                giy += v3 * dxw * go;
            }
        };
        if (p.W >= 2) {
            // The west and east corner of a row are neighbours in memory: one load of two elements (aligned to one
            // element only) per row instead of two loads halves the addresses the gather puts through the memory
            // pipeline.  The pair sits at column pb = clamp(x0, 0, W - 2), so it never leaves the row; which half is
            // which corner follows from pb.  Corners outside the image are skipped by accumulate() as before.
            using PairBits = typename std::conditional<sizeof(T) == 2, uint32_t, uint64_t>::type;
            const int32_t x0 = tp.x0, x1 = (tp.x0 == INT32_MAX) ? tp.x0 : tp.x0 + 1;
            const int32_t y1 = (tp.y0 == INT32_MAX) ? tp.y0 : tp.y0 + 1;
            const int32_t pb = (x0 < 0) ? 0 : ((x0 > p.W - 2) ? p.W - 2 : x0);
            const bool lo_w = (x0 == pb), lo_e = (x1 == pb);
            const int32_t r0 = (tp.y0 >= 0 && tp.y0 < p.H) ? tp.y0 * p.W + pb : 0;
            const int32_t r1 = (y1 >= 0 && y1 < p.H) ? y1 * p.W + pb : 0;
            for_groups([&](auto count, int32_t c) __attribute__((always_inline)) {
                constexpr int U = decltype(count)::value;
                float go[U];
                PairBits north[U], south[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const T* xc = x_n + (int64_t)(c + u) * plane_px;
                    go[u] = ElemIO<T>::load(go_n + (int64_t)(c + u) * points);
                    __builtin_memcpy(&north[u], xc + r0, sizeof(PairBits));
                    __builtin_memcpy(&south[u], xc + r1, sizeof(PairBits));
                }
#pragma unroll
                for (int u = 0; u < U; u++) {
                    T n2[2], s2[2];
                    __builtin_memcpy(n2, &north[u], sizeof(PairBits));
                    __builtin_memcpy(s2, &south[u], sizeof(PairBits));
                    const float nlo = ElemIO<T>::load(&n2[0]), nhi = ElemIO<T>::load(&n2[1]);
                    const float slo = ElemIO<T>::load(&s2[0]), shi = ElemIO<T>::load(&s2[1]);
                    accumulate(go[u], lo_w ? nlo : nhi, lo_e ? nlo : nhi, lo_w ? slo : shi, lo_e ? slo : shi);
                }
            });
        } else {
            for_groups([&](auto count, int32_t c) __attribute__((always_inline)) {
                constexpr int U = decltype(count)::value;
                float go[U], v[U][4];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const T* xc = x_n + (int64_t)(c + u) * plane_px;
                    go[u] = ElemIO<T>::load(go_n + (int64_t)(c + u) * points);
                    v[u][0] = ElemIO<T>::load(xc + o0);
                    v[u][1] = ElemIO<T>::load(xc + o1);
                    v[u][2] = ElemIO<T>::load(xc + o2);
                    v[u][3] = ElemIO<T>::load(xc + o3);
                }
#pragma unroll
                for (int u = 0; u < U; u++) {
                    accumulate(go[u], v[u][0], v[u][1], v[u][2], v[u][3]);
                }
            });
        }
    } else {
        const float xf = __builtin_floorf(tp.fx), yf = __builtin_floorf(tp.fy);
        float cx[4], cy[4], cxg[4], cyg[4];
        cubic_coefficients(cy, tp.fy - yf);
        cubic_coefficients(cx, tp.fx - xf);
        cubic_coefficients_grad(cyg, tp.fy - yf);
        cubic_coefficients_grad(cxg, tp.fx - xf);
        for (int32_t c = 0; c < p.C; c++) {
            const T* xc = x_n + (int64_t)c * plane_px;
            const float go = ElemIO<T>::load(go_n + (int64_t)c * points);
            T v[16];  // all on their way together; a tap outside the plane counts as 0
#pragma unroll
            for (int k = 0; k < 16; k++) {
                v[k] = xc[tp.off[k] >= 0 ? tp.off[k] : 0];
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float w = (tp.off[i * 4 + j] >= 0) ? ElemIO<T>::load(&v[i * 4 + j]) : 0.0f;
                    giy += w * cyg[j] * cx[i] * go;
                    gix += w * cxg[i] * cy[j] * go;
                }
            }
        }
    }
    // products in fp32 first, then the conversion (see contribution())
    ElemIO<T>::store(dgrid + 2 * idx, as_fp32_value(tp.mx * gix));
    ElemIO<T>::store(dgrid + 2 * idx + 1, as_fp32_value(tp.my * giy));
}

struct Grid3Params {
    Grad3Params g;
    int64_t total;  // points of the batch
};

inline Grid3Params grid3_params(const GradGatherArgs& a)
{
    Grid3Params q{};
    q.g.C = (int32_t)a.C;
    q.g.D = (int32_t)a.D;
    q.g.H = (int32_t)a.H;
    q.g.W = (int32_t)a.W;
    q.g.points = (int32_t)a.points;
    q.g.pad = a.pad;
    q.g.align = a.align;
    q.total = a.N * a.points;
    return q;
}

// U: channels whose loads are on their way together (gs3d_point_grid_gradient)
template <typename T, int INTERP, int U>
__device__ __forceinline__ void gs3d_grid_gradient_block(uint32_t block_index, const T* __restrict__ gout, const T* __restrict__ x,
                                                         const T* __restrict__ grid, T* __restrict__ dgrid, const Grid3Params& p)
{
    const int64_t idx = (int64_t)block_index * kChunkPoints3 + threadIdx.x;
    if (idx >= p.total) {
        return;
    }
    if (INTERP == 1) {
        // grid_sampler3_d_grad_simt_det.h:354-356
        ElemIO<T>::store(dgrid + 3 * idx, 0.0f);
        ElemIO<T>::store(dgrid + 3 * idx + 1, 0.0f);
        ElemIO<T>::store(dgrid + 3 * idx + 2, 0.0f);
        return;
    }
    if constexpr (INTERP == 0) {
        const int32_t points = p.g.points;
        const int64_t n = idx / points;
        const int32_t pt = (int32_t)(idx - n * points);
        GradTaps3<T, INTERP> tp;
        decide_grad_taps3<T, INTERP>(tp, ElemIO<T>::load(grid + 3 * idx), ElemIO<T>::load(grid + 3 * idx + 1),
                                     ElemIO<T>::load(grid + 3 * idx + 2), p.g.D, p.g.H, p.g.W, p.g.pad, p.g.align);
        gs3d_point_grid_gradient<T, U>(tp, gout, x, dgrid, idx, n, pt, p.g);
    }
}

}  // namespace opscv
