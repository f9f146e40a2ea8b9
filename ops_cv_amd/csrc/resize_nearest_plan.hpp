// Launch plan of the nearest resize by runs of rows (resize_kernels.hip): host arithmetic only.
#pragma once

#include <cstdint>

#include "acl_types.hpp"
#include "launch_limits.hpp"

namespace opscv {

constexpr int64_t kNearestRowsLds = 60 << 10;   // table, starts and source bytes of a workgroup
constexpr int64_t kNearestRowsOut = 32 << 10;   // output bytes of a workgroup, at the longest run of rows

struct NearestRows {
    int32_t run = 0;  // output rows of a workgroup, a multiple of eight; 0: another kernel
    int32_t cols = 0;  // elements of a row that a workgroup takes, and how many such pieces a row has
    int64_t chunks = 0;
    int64_t rows = 0, blocks = 0;  // of runs
    int64_t lds_bytes = 0, source_bytes = 0;
};

// `in_chunks`: whether the kernel that takes 256 vectors of a row at a time out of LDS can run; it does where its vectors fill
// half of a workgroup.  Shrinking rows reuse nothing, and pixels of whole vectors take one vector load a lane: not here.  Nor
// outputs below a MiB, which are a chain of copy, table and barrier here and one load and store there (fp16 1x6x61x91 ->
// 122x182 5.0 / 6.6, bf16 1x5x117x158 -> 234x316 5.1 / 6.0; 2.4 MB and above: 7.5 / 5.2).
//
// Microseconds before / here (floor at 6 TB/s).  Rows off the 16-byte grid, which were gathered: fp16 6x4x764x1263 -> 1528x2526
// 117 / 42 (39), fp32 17x11x62x120 -> 151x292 20.6 / 8.1 (6.4), channels last fp16 4x1x1004x1749 -> 4016x6996 208 / 42 (40),
// bf16 3x16x613x1196 -> 867x1693 80 / 38 (35).  Narrow rows on it, which left most lanes idle: bf16 15x174x74x83 -> 296x332
// 291 / 121 (91), bf16 3x141x92x80 -> 184x160 39 / 8 (5).  Rows too long to stage whole, in pieces: channels last bf16
// 12x145x92x116 -> 184x232 166 / 35 (31), 6x4x835x1069 -> 1670x2138 162 / 40 (36).
inline NearestRows nearest_rows_plan(const ResizeArgs& a, bool in_chunks)
{
    NearestRows p;
    const int64_t esz = elem_size(a.elem), V = 16 / esz;
    const int64_t ci = a.channels_last ? a.C : 1;
    if (a.mode != ResizeMode::Nearest || a.force_nearest != 0 || a.Hd < a.Hs || a.Wd < a.Ws || (a.channels_last && a.C % V == 0)) {
        return p;
    }
    const int64_t out_row = a.Wd * ci, in_row = a.Ws * ci;
    p.rows = a.N * (a.channels_last ? 1 : a.C) * a.Hd;
    if (p.rows > INT32_MAX / 2 || a.Hd > INT32_MAX / 2 || out_row > INT32_MAX / 128 || in_row * esz > INT32_MAX ||
        (in_chunks && (out_row + V - 1) / V > 96) || p.rows * out_row * esz < (1 << 20)) {
        return p;
    }
    const double last = a.rep_h > 0 ? (double)((a.Hd - 1) / a.rep_h) : (double)((float)(a.Hd - 1) * a.scale_h);
    const int64_t unused = last >= (double)(a.Hs - 1) ? 0 : a.Hs - 1 - (int64_t)last;
    // rows from the first to the last, with those that no row takes at the end of every plane that the run may cross
    auto source_rows = [&](int64_t run) {
        return (int64_t)((double)run * (a.rep_h > 0 ? 1.0 / a.rep_h : (double)a.scale_h) * 1.001) + 2 +
               (run / a.Hd + 1) * (unused + 1);
    };
    auto table = [&](int64_t cols, int64_t run) { return (cols * 2 + 4 * V + 15) / 16 * 16 + run * 4 + 1024; };
    for (int32_t run = 64; run >= 8 && out_row <= 8192 && in_row * esz <= 65535; run /= 2) {
        const int64_t source = source_rows(run) * in_row * esz + 16, lds = table(out_row, run) + source;
        const int64_t blocks = (p.rows + run - 1) / run;
        if (lds <= kNearestRowsLds && ((run * out_row * esz <= kNearestRowsOut && blocks >= 1024) || run == 8) &&
            fits_launch(blocks, 256)) {
            p.run = run;
            p.cols = (int32_t)out_row;
            p.chunks = 1;
            p.blocks = blocks;
            p.lds_bytes = lds;
            p.source_bytes = source;
            return p;
        }
    }
    if (in_chunks) {
        return p;
    }
    p.blocks = (p.rows + 7) / 8;
    if (p.blocks > 65535) {
        return p;
    }
    // Whether a piece of so many vectors fits; shorter ones do where longer ones do, so the longest is searched for by halves
    // (trying one number of pieces after the other took 9 us of host time a call where none fits: channels last, 1001 channels).
    auto bytes = [&](int64_t vectors, int64_t* source) {
        const double factor = a.rep_w > 0 ? 1.0 / a.rep_w : (double)a.scale_w;
        const int64_t segment = (int64_t)((double)(vectors * V) * factor * 1.001) + 3 * ci + 3;
        *source = source_rows(8) * ((segment * esz + 30) / 16 * 16) + 16;
        return segment * esz <= 65535 ? table(vectors * V, 8) + *source : INT64_MAX;
    };
    int64_t most = 0, source = 0;
    for (int64_t low = 1, high = 8192 / V; low <= high;) {
        const int64_t mid = (low + high) / 2;
        const bool fits = bytes(mid, &source) <= kNearestRowsLds / 2;
        most = fits ? mid : most;
        low = fits ? mid + 1 : low;
        high = fits ? high : mid - 1;
    }
    const int64_t chunks = most == 0 ? 0 : (out_row + most * V - 1) / (most * V);
    if (most == 0 || chunks > 1024) {
        return p;
    }
    const int64_t pieces = chunks < 2 ? 2 : chunks;
    const int64_t cols = ((out_row + pieces - 1) / pieces + V - 1) / V * V;
    p.run = 8;
    p.cols = (int32_t)cols;
    p.chunks = (out_row + cols - 1) / cols;
    p.lds_bytes = bytes(cols / V, &source);
    p.source_bytes = source;
    return p;
}

}  // namespace opscv
