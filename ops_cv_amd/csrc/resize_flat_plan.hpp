// How the flat resize (resize_flat_lds_kernel.hpp) walks rows and stores them: host arithmetic only.
#pragma once

#include <cstdint>

#include "acl_types.hpp"

namespace opscv {

constexpr int64_t kFlatPlainBytes = 64ll << 20;   // outputs from here on leave by plain stores
constexpr int64_t kLastLevelBytes = 256ll << 20;  // the chip's last-level cache

struct FlatStores {
    bool streaming = false;  // non-temporal stores
    bool runs = false;       // a row group takes consecutive rows and keeps the blended source rows they share
};

inline FlatStores flat_stores(const ResizeArgs& a)
{
    // Non-temporal stores keep small outputs from lying dirty in L2 at the kernel's end, but write a row's first and last
    // line, which it shares with its neighbours, in pieces.  Non-temporal / plain: fp32 8x64x112x112 (26 MB) 7.0 / 8.9
    // us, bf16 8x256x112x112 (51 MB) 17.4 / 18.6; 8x40x257x513 (84 MB) 26.6 / 23.4, 8x64x257x513 (135 MB) 45.1 / 32.6,
    // fp16 8x512x200x200 (328 MB) 121 / 92, fp32 8x256x112x112 (103 MB) 23.7 / 21.0, 8x32x257x516 (136 MB) 41.7 / 30.1;
    // lines of fp32 rows beyond the last-level cache are better written through: 8x64x257x513 (270 MB) 57.2 / 62.2.
    const int64_t esz = elem_size(a.elem), planes = a.N * a.C;
    const int64_t out_bytes = planes * a.Hd * a.Wd * esz;
    // Beyond the cache, rows of whole vectors keep rows in turn and non-temporal stores, which then fill shared lines
    // together: fp16 8x512x200x200 86 us, 92 otherwise, fp32 8x256x200x200 (328 MB) 82 and 92 (ragged rows bf16
    // 8x256x257x513, 540 MB: 233 and 161).
    // So do fp32 launches of which input and output together are beyond it: in turn and non-temporal / kept and plain, fp32
    // 1x5869x42x65 to 88x114 51.6 / 71.9 us, 1x4273x56x71 to 112x113 51.1 / 60.5 (kept and plain takes 1.13 times the time
    // over 19 launches repeated on the same operands, 1.02 over 26 with operands from memory; 16-bit 0.99 and 0.98).
    const int64_t moved = out_bytes + planes * a.Hs * a.Ws * esz;
    const bool in_turn = (out_bytes >= kLastLevelBytes && (a.Wd * esz) % 16 == 0) ||
                         (out_bytes < kLastLevelBytes && esz == 4 && moved >= kLastLevelBytes);
    FlatStores s;
    s.streaming = out_bytes < kFlatPlainBytes || in_turn || (esz == 4 && out_bytes >= kLastLevelBytes);
    // Rows that grow share source rows: a group's rows are consecutive then, and blended rows are kept (half to an eighth
    // of the LDS reads; with plain stores 33 us on bf16 8x64x65x129 to 257x513, 59 before).
    s.runs = a.Hd > a.Hs && !in_turn;
    return s;
}

}  // namespace opscv
