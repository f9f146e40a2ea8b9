// Plan of the samplers' sorting input gradient (gs_grad_gather.hip), and which of the two ordered variants a launch
// takes: host arithmetic only.
#pragma once

#include <cstdint>

#include "acl_types.hpp"
#include "launch_limits.hpp"

namespace opscv {

// Bytes of scratch.  A batch whose items need more than the first together is run some items at a time, in the same scratch;
// an item that needs more than the second is left to the elections.  The first is the last-level cache's size: fp32
// 64x3x720x1280 in one go (1.4 GiB) 3696 us, in groups of 512 MiB 3798, 256 MiB 3627, 128 MiB 3837, 64 MiB 4380; 16x3x
// 1080x1920 2119 (0.8 GiB), 1969 in groups of 256 MiB; bicubic 8x3x1080x1920 7997 (2.3 GiB), 7662 an item at a time (290 MiB).
constexpr int64_t kGatherGroupScratch = (int64_t)256 << 20;
constexpr int64_t kGatherMostScratch = (int64_t)4 << 30;

struct GradGatherArgs {
    Elem elem = Elem::F32;
    int dim = 2;
    int interp = 0, pad = 0, align = 0;
    int64_t N = 0, C = 0, D = 1, H = 0, W = 0;
    int64_t points = 0;          // grid points per batch item
    int64_t items_per_core = 1;  // batch items whose points are cut into chunks as one run (3-D; 1 for planes)
    const void* gout = nullptr;
    const void* grid = nullptr;
    void* dx = nullptr;
    void* scratch = nullptr;  // grad_gather_words() 32-bit words on a 16-byte boundary
    // the gradient of the grid, for the launches of the input gradient to take along; null: not wanted
    const void* x = nullptr;
    void* dgrid = nullptr;
    int64_t Ho = 0, Wo = 0;   // planes: extents of the grid
};

constexpr int kGatherThreads = 256;
constexpr int kListMost = 32;        // contributions of an element that the gather kernel takes at most
constexpr uint32_t kSortedRun = 64;  // runs of more entries are sorted in place before the crowded kernel reads them
constexpr int kCtrlWords = 16;       // [0] entries handed out, [1] long runs, [2] crowded elements

struct GatherLayout {  // offsets in 32-bit words within an item's scratch
    uint32_t counts;   // behind the control words: cleared together with them
    uint32_t starts;
    uint32_t ranks;    // [entry of a point][point]
    uint32_t coords;   // source coordinates of the points: 2 (4 for volumes) values of the element type
    uint32_t list;     // entries, run after run
    uint32_t runs;     // cells whose run has more than kSortedRun entries
    uint32_t crowded;  // elements with more contributions than their list holds
    uint32_t item_words;
};

struct GatherParams {
    int32_t C, D, H, W, points;
    int32_t pad, align;
    int32_t items_per_core;
    int32_t elements, cells;
    int32_t N;           // items of this launch, and the batch's number of the first one
    int32_t first_item;
    GatherLayout lay;
};

struct GatherPlan {
    bool ok = false;
    GatherParams p{};    // of the first group of items
    int64_t group = 0;   // items run at a time
    uint32_t tiles = 0, cblocks = 0;
    int32_t chans_per_block = 0;
    int cb = 1;
    int list = kListMost;
};

// A list of 16 leaves LDS and registers for twice the wavefronts; of 32 where a smooth grid has more than six
// contributions per element on average (scaled by 0.8 along every axis they are ten)
inline int gather_list(int64_t contributions, int64_t elements)
{
    return contributions <= 6 * elements ? 16 : kListMost;
}

inline uint32_t align4(uint64_t v) { return (uint32_t)((v + 3u) & ~(uint64_t)3u); }

inline GatherPlan gather_plan(const GradGatherArgs& a)
{
    GatherPlan pl;
    const int64_t esz = elem_size(a.elem);
    const int64_t elements = a.D * a.H * a.W;
    const int64_t cells = (a.interp != 0) ? elements : (a.W + 1) * (a.H + 1) * (a.dim == 3 ? a.D + 1 : 1);
    const int64_t entries = a.points * (a.interp == 2 ? 16 : 1);
    const int64_t runs = a.interp == 0 ? ((int64_t)1 << a.dim) : 1;
    // keys of 32 bits hold an entry and a corner; counts of 32 bits hold an item's entries
    const int64_t most_points = (int64_t)1 << (a.dim == 3 || a.interp == 2 ? 27 : 28);
    if (a.points > most_points || elements > INT32_MAX / 2 || cells > INT32_MAX / 2 || a.N > 65535 || a.N < 1) {
        return pl;
    }
    pl.list = gather_list(entries * runs, elements);
    const int64_t crowded_elements = entries * runs / (pl.list + 1) + 1;
    const int64_t words = kCtrlWords + 2 * cells + 2 * entries + a.points * (a.dim == 3 ? 4 : 2) * esz / 4 +
                          entries / kSortedRun + crowded_elements + 64;
    if (words > ((int64_t)1 << 31) || words * 4 > kGatherMostScratch) {
        return pl;
    }
    const int64_t fit = kGatherGroupScratch / (words * 4);
    const int64_t group = fit < 1 ? 1 : (fit < a.N ? fit : a.N);
    pl.group = (a.N + (a.N + group - 1) / group - 1) / ((a.N + group - 1) / group);  // as many items in every group
    GatherLayout& l = pl.p.lay;
    l.counts = kCtrlWords;
    l.starts = align4((uint64_t)l.counts + (uint64_t)cells);
    l.ranks = align4((uint64_t)l.starts + (uint64_t)cells);
    l.coords = align4((uint64_t)l.ranks + (uint64_t)entries);
    l.list = align4((uint64_t)l.coords + (uint64_t)(a.points * (a.dim == 3 ? 4 : 2) * esz / 4));
    l.runs = align4((uint64_t)l.list + (uint64_t)entries);
    l.crowded = align4((uint64_t)l.runs + (uint64_t)(entries / kSortedRun) + 1u);
    l.item_words = align4((uint64_t)l.crowded + (uint64_t)crowded_elements);
    pl.p.C = (int32_t)a.C;
    pl.p.D = (int32_t)a.D;
    pl.p.H = (int32_t)a.H;
    pl.p.W = (int32_t)a.W;
    pl.p.points = (int32_t)a.points;
    pl.p.pad = a.pad;
    pl.p.align = a.align;
    pl.p.items_per_core = (int32_t)(a.items_per_core > 0 ? a.items_per_core : 1);
    pl.p.elements = (int32_t)elements;
    pl.p.cells = (int32_t)cells;
    pl.p.N = (int32_t)pl.group;
    pl.p.first_item = 0;
    pl.cb = (a.C >= 8) ? 8 : ((a.C >= 3) ? 4 : (int)a.C);
    pl.tiles = (uint32_t)((elements + kGatherThreads - 1) / kGatherThreads);
    const int64_t base = pl.group * pl.tiles;
    const int64_t max_cblocks = (a.C + pl.cb - 1) / pl.cb;
    int64_t cblocks = (2048 + base - 1) / base;
    cblocks = cblocks > max_cblocks ? max_cblocks : cblocks;
    int64_t cpb = (a.C + cblocks - 1) / cblocks;
    cpb = (cpb + pl.cb - 1) / pl.cb * pl.cb;
    cblocks = (a.C + cpb - 1) / cpb;
    pl.cblocks = (uint32_t)cblocks;
    pl.chans_per_block = (int32_t)cpb;
    pl.ok = fits_launch(base * cblocks + 8 + 65536, kGatherThreads) &&  // padded to the XCDs, and the sorting workgroups
            fits_launch(pl.group * ((a.points + kGatherThreads - 1) / kGatherThreads) + 8, kGatherThreads);
    return pl;
}

// Microseconds of the input gradient of planes by either variant, from sizes alone (the kernels' device time also
// depends on how evenly a grid spreads its points).
//
// Elections: `chunks` steps one after the other, a turn of the chip (1024 workgroups) after the other; a step's election
// takes a round more where a chunk's points share elements.  Sorting: passes over elements, contributions and their
// channels, and again over the contributions of elements that hold more than a list, where a wavefront folds in order.
// Fitted to 4200 calls of both (1 to 600 items, 1 to 200 channels, planes of 16 to 10^6 elements, 0.005 to 30 points per
// element, turned and scattered grids, 5 us to 15 ms): half of the estimates are within 20 percent of the time, nine of
// ten between half of it and half as much again.
struct PlaneGradTimes {
    double elections, sorting;
};

inline PlaneGradTimes plane_grad_times(const GradGatherArgs& a)
{
    struct Rates {
        double e_call, e_chunk, e_turn, e_band, e_shared, e_groups;                             // elections
        double s_call, s_element, s_entry, s_value, s_store, s_crowded, s_crowded_value, s_chain, s_run;  // sorting
    };
    static const Rates kRates[3] = {
        {2.9, 0.43, 1.6, 3.0, 0.22, 2.7, 20.0, 12.0, 10.0, 3.3, 0.81, 35.0, 2.0, 0.47, 17.0},   // bilinear
        {5.6, 0.014, 0.93, 0.66, 0.087, 0.85, 18.0, 9.8, 38.0, 4.5, 0.99, 26.0, 1.9, 1.0, 7.0},  // nearest
        {1.1, 3.3, 8.7, 5.5, 1.9, 3.8, 30.0, 15.0, 33.0, 1.6, 0.78, 28.0, 2.0, 0.35, 3.5},       // bicubic
    };
    const Rates& r = kRates[a.interp];
    const double M = 1e-6;
    const double elements = (double)(a.H * a.W), points = (double)a.points, N = (double)a.N, C = (double)a.C;
    auto least = [](double u, double v) { return u < v ? u : v; };
    PlaneGradTimes t;

    const int64_t group = 8 / elem_size(a.elem);  // channels of an election workgroup; fewer run one per workgroup
    const double groups = (double)(a.C >= group ? (a.C + group - 1) / group : a.C);
    const double band = least(elements, 4096.0);
    const double workgroups = (double)((int64_t)((elements + band - 1) / band)) * groups * N;
    const double turns = workgroups > 1024.0 ? workgroups / 1024.0 : 1.0;
    const double chunks = (double)((a.points + 255) / 256);
    t.elections = r.e_call + chunks * (r.e_chunk + turns * (r.e_turn + band / elements *
                  (r.e_band + r.e_shared * least(256.0, points / elements)))) + r.e_groups * workgroups / 1024.0;

    const double taps = (a.interp == 0) ? 4.0 : ((a.interp == 1) ? 1.0 : 16.0);
    const double contributions = taps * points, entries = (a.interp == 2) ? contributions : points;
    // from 0.4 of a list per element on average some hold more than one, from a whole list on all do; likewise for runs
    const double list = gather_list((int64_t)contributions, (int64_t)elements);
    auto ramp = [&](double v, double from) { return v <= from ? 0.0 : least(1.0, (v - from) / (1.0 - from)); };
    const double crowded = ramp(contributions / elements / list, 0.4);
    const double runs = ramp(entries / elements / kSortedRun, 0.5);
    t.sorting = r.s_call + N * M * (r.s_element * elements + r.s_entry * contributions + C * (r.s_value * contributions +
                r.s_store * elements) + crowded * contributions * (r.s_crowded + r.s_crowded_value * C)) +
                r.s_chain * crowded * contributions / elements + r.s_run * runs * N * elements * 1e-3;
    return t;
}

// Whether the sorting variant takes the input gradient of planes (where the list variant does not).  The rates above and the
// figures below are of sorting by lists (gs_grad_gather.hip).  Where the tiles of gs_grad_tiles.hip take the call sorting is up
// to twice as fast, so the lines lie on the elections' side there: some calls near them would be faster sorted.
//
// Up to 24 tap passes over a chunk (6 chunks bilinear, 24 nearest, 1 bicubic) the elections take 10 to 30 us and sorting as
// much or more.  Sorting against elections over grids and planes of up to eight items, medians: bilinear 5 and 6 chunks
// 0.95, 7 and 8 0.52; nearest 13 to 16 1.05, 17 to 24 0.90, 25 to 30 0.82; bicubic 1 chunk 1.69, 2 0.95, 3 0.74 (fp32 N1 C3:
// bilinear 4 chunks 17 us against 20, 9 chunks 32 / 22; bicubic 1 chunk 24 / 36, 3 chunks 50 / 41).  Beyond, sorting
// wins unless batches are large (every item costs its passes over the plane, the elections of a thousand workgroups run
// side by side) or points are few on large planes, or many on small ones: fp32 512 x 3 x 64x64 from 40x40 points 24.9 us
// against 75.6, 1 x 3 x 1080x1920 from 40x40 18.3 / 57.6, 1024 x 1 x 16x16 from 64x64 100 / 1014; bicubic 512 x 3 x
// 64x64 340 / 1682.  The elections' time follows the grid more than sorting does (a chunk of a turned grid on a small
// plane can take three times the rounds of a scattered one), nearest samples' most: hence the margins, which leave a launch
// to sorting unless the elections are clearly faster.  Of the 1970 calls that sorting would take by tap passes alone, 237 were
// slower than elections, the worst 8.7 times; with the estimates 93, the worst but one (7.6 times: long runs of scattered
// bicubic points) 3.1, and 23 of those left to the elections would have been faster sorted, by 2.9 at most.
inline bool sorting_takes_planes(const GradGatherArgs& a)
{
    const int64_t chunks = (a.points + 255) / 256;
    const int64_t taps = (a.interp == 0) ? 4 : ((a.interp == 1) ? 1 : 16);
    if (chunks * taps <= 24) {
        return false;
    }
    const PlaneGradTimes t = plane_grad_times(a);
    const double margin = (a.interp == 1 && a.N < 64) ? 0.5 : 0.7;
    return t.elections >= margin * t.sorting;
}

}  // namespace opscv
