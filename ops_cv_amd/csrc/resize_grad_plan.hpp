// Launch plans of the resize gradient's LDS kernels (resize_grad.hip): host arithmetic only.
#pragma once

#include <cstdint>

#include "acl_types.hpp"
#include "fast_div.hpp"
#include "launch_limits.hpp"

namespace opscv {

constexpr int kGradThreads = 256;

// ---- resize_grad_lds_kernel ----
constexpr int kGradTileCols = 128;
constexpr int64_t kWantBlocks = 8192;
constexpr int32_t kGradCapWords = 12288;  // at most 48 KB of LDS per workgroup (fp32 words, one per tile element)
constexpr int kGradTileGroups = kGradThreads / kGradTileCols;  // row groups of a workgroup

// Output rows per workgroup for the LDS variant (0: use the gather kernel).  The estimate only sizes the launch;
// the kernel measures the rectangle itself.
inline int32_t lds_tile_rows(const ResizeGradArgs& a, int32_t cap_words, int32_t* need_words = nullptr)
{
    const int epw = 4 / elem_size(a.elem_in);
    const int64_t ci = a.channels_last ? a.C : 1;  // row elements per pixel
    if (a.user_scales || (a.Wd * ci) % epw != 0 || reinterpret_cast<uintptr_t>(a.x) % 4 != 0 ||
        a.Ws * ci > INT32_MAX || a.Wd * ci > INT32_MAX) {
        return 0;
    }
    const double per_col = (double)a.Wd / (double)a.Ws, per_row = (double)a.Hd / (double)a.Hs;
    // a tile of kGradTileCols outgoing elements visits that many times per_col incoming ones, plus two pixels either side
    const double cols = kGradTileCols * per_col + (2.0 * per_col + 2.0) * (double)ci + epw;
    for (int32_t rows = 8; rows >= kGradTileGroups; rows /= 2) {
        const double need = (rows * per_row + 2.0 * per_row + 2.0) * cols;  // fp32 words: one per element
        if (need <= (double)cap_words) {
            if (need_words != nullptr) {
                *need_words = (int32_t)need + 1;
            }
            return rows;
        }
    }
    return 0;
}

struct LdsTile {
    int32_t rows = 0;      // 0: the variant does not apply
    int32_t lds_words = 0;
    int64_t tiles_x = 0, tiles_y = 0;
    int64_t slots = 0;     // workgroups per tile; each takes every slots-th plane
    int64_t blocks = 0;    // padded for the XCD mapping of the kernel
};

inline LdsTile lds_tile(const ResizeGradArgs& a)
{
    LdsTile t;
    const int32_t rows = lds_tile_rows(a, kGradCapWords, &t.lds_words);
    if (rows <= 0) {
        return t;
    }
    // the allocation follows the estimate so that more workgroups share a CU (their load and compute phases overlap);
    // a rectangle that turns out larger than the estimate is read from global memory by the kernel
    t.lds_words = (t.lds_words + 63) / 64 * 64;
    t.lds_words = t.lds_words < kGradCapWords ? t.lds_words : kGradCapWords;
    const int64_t planes = a.channels_last ? a.N : a.N * a.C, row_elems = a.Ws * (a.channels_last ? a.C : 1);
    t.tiles_x = (row_elems + kGradTileCols - 1) / kGradTileCols;
    t.tiles_y = (a.Hs + rows - 1) / rows;
    // A workgroup walks over several planes with the tile geometry and column weights it computed once; enough
    // workgroups are launched to keep every CU supplied (kWantBlocks), the rest of the planes are looped over.
    const int64_t tiles = t.tiles_x * t.tiles_y;
    t.slots = (kWantBlocks + tiles - 1) / tiles;
    t.slots = t.slots < planes ? t.slots : planes;
    t.slots = t.slots < 65535 ? t.slots : 65535;
    t.blocks = (tiles * t.slots + 7) / 8 * 8;
    t.rows = (t.tiles_y <= 65535 && fits_launch(t.blocks, kGradThreads)) ? rows : 0;
    return t;
}

// ---- resize_grad_planes_kernel ----
constexpr int kPlaneCols = 64;
constexpr int kPlaneVisits = 8;                 // most rows, and most columns, an outgoing element may visit
constexpr int kPlaneRows = 16;                  // most outgoing rows of a tile
constexpr int32_t kPlaneTallBytes = 24 * 1024;  // tiles of 16 rows up to here: six workgroups and more fit a CU
constexpr int32_t kPlaneMostBytes = 48 * 1024;  // tiles of 8 rows up to here
constexpr int32_t kPlanePad = 64;               // bytes behind the last row that a lane's last columns may be read from

struct PlaneTile {
    int32_t rows = 0;  // 0: the variant does not apply
    int32_t lds_bytes = 0;
    int64_t tiles_x = 0, tiles_y = 0;
    int64_t slots = 0;   // workgroups per tile; each takes every slots-th plane
    int64_t blocks = 0;  // padded for the XCD mapping of the kernel
    int32_t strip_cols = 0;    // columns past the last whole tile, 0: they are a tile
    int64_t strip_blocks = 0;  // workgroups of them, ahead of the tiles' and counted in blocks
};

// Rows off the word grid go to the planes kernel or to the gather, whichever is estimated to be faster.  The gather's time
// follows the elements and the bytes; the planes kernel's the tiles, whole ones also where planes are narrower than 64
// columns or lower than the tile, and a set-up per turn of the chip: fp16 131072 planes of 3x3 from 7x7 19 us in the
// gather, 142 in tiles; 16384 of 20x5 from 41x11 25 / 136; 16384 of 14x14 from 29x29 46 / 73; bf16 512 of 65x129 from
// 257x513 189 / 72.  Fitted to 1777 launches (1 to 60000 planes of 2 to 2000 columns, 4 to 450 us): of these, 958 were
// slower in tiles than in the gather, by up to 11 times; 92 are with the estimates, by 1.7 at most, and 10 that are left
// to the gather would have been faster in tiles, by 1.2 at most.
inline bool gather_takes_planes(const ResizeGradArgs& a, const PlaneTile& t)
{
    const double planes = (double)(a.N * a.C), elements = planes * (double)a.Hs * (double)a.Ws * 1e-6;
    const double megabytes = elem_size(a.elem_in) * (elements + planes * (double)a.Hd * (double)a.Wd * 1e-6);
    const double tiles = (double)(t.tiles_x * t.tiles_y) * planes * 1e-3;
    const double turns = t.blocks > 1500 ? (double)t.blocks / 1500.0 : 1.0;
    const double rows_visited = 2.0 / (double)a.scale_h, columns = 2.0 / (double)a.scale_w;
    const double visits = t.rows * rows_visited * (columns < kPlaneVisits ? columns : (double)kPlaneVisits);
    const double gather_us = 5.0 + 1.0 * elements + 1.14 * megabytes;
    const double tiles_us = 3.1 + 4.1 * turns + tiles * (0.47 + 0.0038 * visits) + 0.33 * megabytes;
    return gather_us < tiles_us;
}

// Eight visits a side at most (growth by up to four), elements anywhere.  The estimate of the rectangle sizes the
// launch; the kernel measures it and reads a larger one from global memory.
inline PlaneTile plane_tile(const ResizeGradArgs& a)
{
    PlaneTile t;
    const int esz = elem_size(a.elem_in);
    if (a.user_scales || (a.channels_last && a.C != 1) || !(a.scale_h >= 0.25f) || !(a.scale_w >= 0.25f) ||
        reinterpret_cast<uintptr_t>(a.x) % (uintptr_t)esz != 0) {
        return t;
    }
    // resize_grad_lds_kernel spends fewer instructions on a visit and sets a tile up once for many planes: fp16 64 planes
    // of 1080x1920 from 2160x3840 (sixteen planes a workgroup) 405 us there, 452 here.  Below four planes a workgroup this
    // kernel takes 0.60 to 0.78 of that one's time (medians of 576 launches; 1.2 at worst), from four on 0.74 to 0.82 and
    // 1.4 at worst: those launches stay there.  It takes rows on the word grid; above growth by about 2.6 its tiles get
    // lower than 8 x 128 and read too much twice.
    const int64_t wide_tiles = ((a.Ws + kGradTileCols - 1) / kGradTileCols) * ((a.Hs + 7) / 8);
    if (wide_tiles * a.N * a.C >= 4 * kWantBlocks && lds_tile_rows(a, kGradCapWords) == 8) {
        return t;
    }
    const int64_t planes = a.N * a.C;
    const double per_col = 1.0 / (double)a.scale_w, per_row = 1.0 / (double)a.scale_h;
    // a tile visits per_col incoming columns for each of its own and two more a side, and a segment is rounded out
    const double pitch = ((kPlaneCols + 2.0) * per_col + 2.0) * esz + 30.0;
    t.tiles_x = (a.Ws + kPlaneCols - 1) / kPlaneCols;
    for (const int32_t rows : {16, 8}) {
        const double bytes = ((rows + 2.0) * per_row + 2.0) * pitch + kPlanePad;
        t.tiles_y = (a.Hs + rows - 1) / rows;
        if (bytes <= (rows == 16 ? kPlaneTallBytes : kPlaneMostBytes) &&
            (rows == 8 || t.tiles_x * t.tiles_y * planes >= 1024)) {
            t.rows = rows;
            t.lds_bytes = ((int32_t)bytes + 64) / 64 * 64;
            break;
        }
    }
    // a workgroup walks over several planes, all of them as many, with the geometry and weights it computed once
    const int64_t want_blocks = 4096;  // 2048: within 2 us; 8192: 6 us slower where planes are small
    const int64_t tiles = t.tiles_x * t.tiles_y;
    t.slots = (want_blocks + tiles - 1) / tiles;
    t.slots = t.slots < planes ? t.slots : planes;
    const int64_t walk = (planes + t.slots - 1) / t.slots;
    t.slots = (planes + walk - 1) / walk;
    t.blocks = (tiles * t.slots + 7) / 8 * 8;
    if (!fits_launch(t.blocks, kGradThreads)) {  // tall planes of a few columns: the gather walks its elements
        t.rows = 0;
    }
    if (t.rows > 0 && lds_tile_rows(a, kGradCapWords) == 0 && gather_takes_planes(a, t)) {
        t.rows = 0;
    }
    // Columns past the last whole tile.  A tile spends a wavefront on every row of them, however few; read in place they cost a
    // lane per element.  Microseconds as a tile / a lane per element, 512 planes of 64 rows:
    //   past the first tile (half of the launch's tiles): growth by 0.7, 1.4, 2, 3 and 4, 16 columns, bf16 18.1 / 14.6,
    //   24.9 / 19.9, 30.0 / 24.4, 49.6 / 38.6, 50.1 / 44.4, fp32 17.5 / 14.0, 24.2 / 19.2, 29.2 / 23.7, 43.0 / 38.9,
    //   87.9 / 79.6; 24 columns, growth by 4 50.3 / 57.4 and 88.8 / 95.1;
    //   past the fourth: 0.7 and 1.4, 16 columns, bf16 26.7 / 25.5, 41.6 / 38.9, fp32 25.9 / 24.5, 40.4 / 38.2, 24 columns
    //   41.1 / 42.4; growth by 2, 8 columns, 51.9 / 45.7 and 50.6 / 48.2, 12 columns, fp32 50.8 / 52.0; growth by 3, 6 columns,
    //   fp32 85.5 / 87.6.
    // bf16 512 planes of 65x129 from 257x513 72 / 55.  Few planes are 0 to 15 % faster, 24 growing by 2 and one column 6.2 / 5.7,
    // but for growth by four with few elements, whose chain of eight rows outlasts the tiles: 24 of 64x65 9.0 / 9.5, of 64x257
    // 12.0 / 12.9, with 64x72 (12288 elements) 8.7 / 8.2.
    const int64_t rest = a.Ws % kPlaneCols, strip = planes * a.Hs * rest;
    const double visits = 4.0 / ((double)a.scale_h * (double)a.scale_w);  // of an outgoing element
    const int64_t most = (a.Ws < 2 * kPlaneCols || visits <= 8.2) ? 16 : (visits <= 16.5 ? 8 : 4);
    if (t.rows > 0 && a.Ws > kPlaneCols && rest > 0 && rest <= most && planes <= INT32_MAX && strip <= INT32_MAX &&
        (visits <= 40.0 || strip >= 12288)) {
        PlaneTile s = t;
        s.strip_cols = (int32_t)rest;
        s.strip_blocks = ((strip + kGradThreads - 1) / kGradThreads + 7) / 8 * 8;
        s.tiles_x = a.Ws / kPlaneCols;
        s.blocks = (s.tiles_x * s.tiles_y * s.slots + 7) / 8 * 8 + s.strip_blocks;
        t = fits_launch(s.blocks, kGradThreads) ? s : t;
    }
    return t;
}

// ---- resize_grad_rows_kernel ----
// Most columns, and most rows, an outgoing element may visit: 2 / scale, and one more at growth by a whole number, where
// coordinates meet on both ends and their rounding decides.  Growth by five: eleven for one element in two to five.  (A wavefront
// that meets more goes down its columns from memory, a lane each: with ten here fp32 4 planes of 64x64 20.4 us, now 7.9, 256 of
// 14x14 22.7 / 8.6, fp16 16 of 100x100 22.6 / 9.6, by the kernels above 11.2, 12.5, 15.2.)
constexpr int kRowsColumns = 12;
constexpr float kRowsLeastScale = 0.2f;

constexpr int64_t kRowsMost = 1 << 18;    // outgoing rows: single precision tells which of them visit a row, but for neighbours

struct RowsPlan {
    bool ok = false;
    uint32_t columns = 0;  // of all planes, side by side
    FastDiv by_ws, by_groups;
    bool two = false;      // a row of a wavefront's columns may have more than 64 units of 16 bytes
    int visits = 8;        // rows that an element may visit: 8, 10 or 12, and columns: 10, or 12 where the rows are 12
    int32_t rows = 0;      // outgoing rows of a wavefront
    int64_t blocks = 0;    // padded for the XCD mapping of the kernel
};

// Planes that grow by up to five.  Left to the kernels above: more than 2^18 rows; planes of 1 GiB and more, or, of fewer than 64
// columns, of 2 GiB over the planes that a wavefront may reach (span); up to three columns of fewer than 2^19 elements; and rows whose
// units of 16 bytes are estimated at more than two a lane.  That estimate counts whole planes where a wavefront has 64 columns
// of them, some of which it cuts: fp32 planes of 55 to 63 columns that grow by three, 48 to 63 by 3.5, 42 to 63 by four, 28 to 63 by 4.5
// are left although what they load fits (71 units at most by four).
// Against them, medians of three runs, device time in microseconds before / with it: bf16 8x64x65x129 from 257x513 58 / 44, fp32 81 / 57,
// fp16 64x128 from 256x512 53 / 41; growth by two fp32 4x16x270x480 43 / 32, fp16 16x64x56x56 29 / 17, 4x16x1080x1920 437 / 415, bf16
// 512x32x14x14 43 / 17; growth by 1.1 fp32 2000 planes of 82x424 315 / 164, fp16 182 / 143; shrunk by 0.5 120 / 104 and 30 / 29 (64
// planes of 400x600), by 0.35 28 / 28.  Growth by four with aligned corners, where an element visits nine rows and columns: fp16 85
// planes of 539x108 206 (tiles of two rows in LDS) / 54.8.  Over 260 random shapes (1 to 20000 planes of 2 to 1500 columns, growth by
// 0.25 to 4) 1.57 times as fast, none slower by more than a microsecond.
inline RowsPlan rows_plan(const ResizeGradArgs& a)
{
    RowsPlan r;
    const int esz = elem_size(a.elem_in);
    const int64_t planes = a.N * a.C;
    if (a.user_scales || (a.channels_last && a.C != 1) || !(a.scale_h >= kRowsLeastScale) || !(a.scale_w >= kRowsLeastScale) ||
        reinterpret_cast<uintptr_t>(a.x) % (uintptr_t)esz != 0 || planes <= 0 || a.Ws <= 0 || a.Hs <= 0 ||
        planes > INT32_MAX / a.Ws || a.Hs > kRowsMost) {
        return r;
    }
    // Few elements of planes of a column or two spend longer on finding their runs than the gather does on all of it.
    if (a.Ws < 4 && planes * a.Hs * a.Ws < (int64_t)1 << 19) {
        return r;
    }
    // a lane's plane lies up to that far behind the first lane's: 32 bits
    const int64_t span = a.Ws >= 64 ? 2 : 63 / a.Ws + 2;
    if (a.Hd * a.Wd > INT32_MAX / (span * esz)) {
        return r;
    }
    // units of a row: of whole planes, or of a run that the end of a plane may cut
    const int64_t units = a.Ws < 64 ? (a.Wd * esz + 30) / 16 * (64 % a.Ws == 0 ? 64 / a.Ws : span)
                                    : (int64_t)((64.0 / a.scale_w + 12.0) * esz + 60.0) / 16;
    if (units > 128) {
        return r;
    }
    r.two = units > 64;
    r.columns = (uint32_t)(planes * a.Ws);
    r.by_ws = make_fast_div((uint32_t)a.Ws);
    const int64_t tiles = ((int64_t)r.columns + kGradThreads - 1) / kGradThreads;
    // a kernel for 12 columns takes seven registers more, and a wavefront of six off a SIMD: fp16 4x16x1080x1920 by two 425 us by that of
    // 10, 453 by one for all; fp32 2000 planes of 82x424 by 1.1 165 / 180
    const bool five = a.scale_h < 0.2002f || a.scale_w < 0.2002f;
    r.visits = five ? kRowsColumns : (a.scale_h < 0.2501f ? 10 : 8);
    r.rows = 8;
    while (r.rows > 2 && tiles * ((a.Hs + r.rows - 1) / r.rows) < 512) {
        r.rows /= 2;
    }
    // Rows of a wavefront: few enough to fill the chip, as many as leave its workgroups turns to even out (64 and 18 rows of 82
    // took 155 us where 41 and 41 take 104), more of them where a row is soon done (64 planes of 400x600 by 0.5 31 / 29)
    const int64_t enough = a.scale_h > 1.2f ? 1536 : 4096;
    while (r.rows < 64 && r.rows < a.Hs && tiles * ((a.Hs + 2 * r.rows - 1) / (2 * r.rows)) >= enough) {
        r.rows *= 2;
    }
    const int64_t groups = (a.Hs + r.rows - 1) / r.rows;
    r.rows = (int32_t)((a.Hs + groups - 1) / groups);
    r.by_groups = make_fast_div((uint32_t)groups);
    r.blocks = (tiles * groups + 7) / 8 * 8;
    r.ok = fits_launch(r.blocks, kGradThreads);
    return r;
}

// ---- the kernel of a call ----
enum class ResizeGradKernel { Scales, Rows, Planes, Lds, Gather };

struct ResizeGradPlan {
    ResizeGradKernel kernel = ResizeGradKernel::Gather;
    RowsPlan rows;
    PlaneTile planes;
    LdsTile lds;
};

// Few elements that visit few: done before a wavefront of the rows kernel has its weights and its first rows, by a lane an
// element of the gather.  Rows / gather in graphs of 64 calls, microseconds: bf16 49 planes of 10x20 from 11x23 3.9 / 2.5, 35 of 21x187
// from 31x281 4.5 / 3.9, fp16 83 of 8x36 from 6x29 3.6 / 2.4, 144 of 9x196 from 11x245 4.7 / 4.0, fp32 7 of 51x51 from 56x57 3.9 / 2.9,
// 125 of 14x70 by two 4.6 / 4.1, bf16 622 of 45x5 from 91x11 6.1 / 5.0, 4 of 32x18 by 2.5 4.7 / 4.1, fp16 25 of 127x137 by 0.6 4.8 / 4.2;
// beyond fp16 421 of 9x62 by two 5.0 / 5.0, 960 of 3x173 from 3x191 4.9 / 5.2, bf16 477 of 6x123 from 10x215 5.4 / 6.0, fp32 3171 of
// 3x32 from 6x65 5.9 / 6.1, 20 of 116x284 by 1.25 6.1 / 7.2, by 2.5 fp16 2 of 145x132 5.0 / 5.0, 55 of 61x69 5.9 / 7.1.
inline bool gather_takes_few(const ResizeGradArgs& a)
{
    const double elements = (double)a.N * (double)a.C * (double)a.Hs * (double)a.Ws;
    const double visits = 4.0 / ((double)a.scale_h * (double)a.scale_w);  // of an outgoing element
    return elements <= 450e3 && ((visits <= 18.5 && elements * visits <= 3e6) || (visits <= 26.0 && elements * visits <= 0.95e6));
}

inline ResizeGradPlan resize_grad_plan(const ResizeGradArgs& a)
{
    ResizeGradPlan p;
    if (a.user_scales) {
        p.kernel = ResizeGradKernel::Scales;
    } else if (p.rows = rows_plan(a); p.rows.ok) {
        p.kernel = gather_takes_few(a) ? ResizeGradKernel::Gather : ResizeGradKernel::Rows;
    } else if (p.planes = plane_tile(a); p.planes.rows > 0) {
        p.kernel = ResizeGradKernel::Planes;
    } else if (p.lds = lds_tile(a); p.lds.rows > 0) {
        p.kernel = ResizeGradKernel::Lds;
    }
    return p;
}

}  // namespace opscv
