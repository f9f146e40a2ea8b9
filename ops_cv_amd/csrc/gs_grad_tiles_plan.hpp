// Plan of the samplers' input gradient by tiles (gs_grad_tiles.hip): host arithmetic only.
#pragma once

#include <cstdint>

#include "fast_div.hpp"
#include "gs_grad_gather_plan.hpp"

namespace opscv {

constexpr int kBinThreads = 256;
constexpr int kBinPoints = 1024;  // grid points of a block: a segment holds the points of a block that fall on a tile

// A tile of the plane or volume, a lane of a workgroup per element, and the points that the workgroup has in LDS at a time:
// a whole segment at least.
template <int DIM>
struct GradTile;
template <>
struct GradTile<2> {
    static constexpr int kX = 32, kY = 16, kZ = 1;
    static constexpr int kPartX = 8, kPartY = 4, kPartZ = 1;  // of a crowded tile
    static constexpr int kThreads = kX * kY * kZ;
    static constexpr int kRecords = 1024;
};
template <>
struct GradTile<3> {
    static constexpr int kX = 16, kY = 8, kZ = 4;
    static constexpr int kPartX = 4, kPartY = 4, kPartZ = 4;
    static constexpr int kThreads = kX * kY * kZ;
    static constexpr int kRecords = 1280;
};

// A record: the point's number within its block, and above it the part of the tile that its low corner lies in (of the corners
// inside the tile, along every axis) and along which axes its high corner lies in the next part.
constexpr int kRecordBits = 10;
constexpr int kRecordPartBits = 4;  // of the part; an axis a bit each above them

struct TilesLayout {   // offsets in 32-bit words within an item's scratch
    uint32_t segments; // [block][tile]: first record in the block's records, and how many << 16
    uint32_t records;  // [block]: 16-bit records of points, segment after segment
    uint32_t block_words;  // of records
    uint32_t item_words;
};

// Tiles that are left to gs_tiles_crowded_kernel: of more than `points` points, or with an element of more than
// `contributions` among the tile's first points.
//
// The kernel costs a launch, and 4.6 us where no tile is crowded.  Input gradient alone, as many points as elements on a part of
// either axis; lists / rounds of the gather kernel alone / here, microseconds.  Half of an axis stays with the rounds: fp32
// 1x3x480x640 93 / 62 / 64 (112 with every tile beyond one round here), fp16 8x4x256x256 from 360x360 175 / 143 / 146 (225 from
// 3072 points on), nearest 1x3x480x640 34 / 25 / 27 (84).  A quarter: 1x3x480x640 125 / 335 / 80, 8x3x479x637 758 / 372 / 470,
// fp16 2x16x200x300 88 / 332 / 90 (127 from 5120 points on), fp32 2x64x200x200 163 / 589 / 228; nearest 60 / 102 / 102 and 233 /
// 130 / 130 (389 from 4096 on).  An eighth: 167 / 1583 / 151, 820 / 1653 / 388, 120 / 1377 / 124, 218 / 1995 / 184, nearest 86 /
// 529 / 186 and 394 / 563 / 411.  Volumes: fp16 2x4x32x64x64 half 296 / 236 / 92, quarter 487 / 2197 / 252, eighth 1608 / 35542 /
// 1249; fp32 4x16x16x64x64 reflection 339 / 360 / 371 (548 by the line of few channels), 553 / 2712 / 770, 1576 / 30692 / 646;
// nearest 2x4x32x64x64 38 / 33 / 36, 78 / 311 / 194, 119 / 1902 / 633: nearest samples of an eighth of every axis are what the
// lists remain much faster at.  Nine points of ten on five spots: 1x3x480x640 6156 / 2138 / 1433.
// Border padding piles points up on few elements, which the gather kernel's wavefronts add together: no limit of contributions
// (fp16 8x4x256x256 from 360x360 131 / 97 / 100, with the limit 133).  Volumes' borders have elements of 50 to 90 here and
// there, which the gather kernel's wavefronts put in order by counting: gradients with a limit of 48 / 96 / 192 / none, fp16
// reflection 11x2x42x18x88 119 / 97 / 97 / 97, bf16 border 3x4x24x61x31 59 / 51 / 52 / 52.  But border padding piles affine grids
// up on all of a face, whose tiles outlast the launch unless there is other work, and then few elements of points at random:
// limit of 48 / 96 over 40 borders of up to 48 items times channels, affine 1.36 times as fast with 48, near the identity 1.01, at
// random 0.89 (fp32 3x4x40x16x17 62 / 174, 1x10x19x48x26 78 / 138, at random fp16 10x3x16x38x38 99 / 64); 72 / 96 over 13 of up to
// 150 1.13, 0.97 and 1.01 (24x6x22x22x10 102 / 151); reflection, 38 calls, 1.02, 0.97 and 0.89 (fp16 3x6x21x67x39 at random 163 / 104).
struct CrowdedTile {
    uint32_t points, contributions;
};
inline CrowdedTile crowded_tile(const GradGatherArgs& a)
{
    const uint32_t any = 0xFFFFFFFFu;
    if (a.interp == 1) {
        return {a.dim == 3 ? 10240u : 12288u, any};
    }
    if (a.dim == 3) {
        const bool few = a.N * a.C <= 48;
        return {few ? 1920u : 6144u, a.pad != 1 ? 96u : (few ? 48u : 72u)};
    }
    return {a.C > 8 ? 3072u : 5120u, a.pad == 1 ? any : 48u};
}

struct TilesParams {
    int32_t C, D, H, W, points;
    int32_t pad, align;
    int32_t items_per_core;
    int32_t elements;
    int32_t N;  // items of this launch, and the batch's number of the first one
    int32_t first_item;
    int32_t tiles_x, tiles_y, tiles;
    int32_t blocks;  // of points
    FastDiv by_tiles_x, by_tiles_y, by_tiles, by_blocks, by_item;  // the last: workgroups of the gather kernel per item
    TilesLayout lay;
    // crowded tiles: which, how many there can be in the launch, and where in scratch their list is (how many there are, then
    // item << kTileBits | tile of each)
    CrowdedTile crowded;
    uint32_t list_most, list;
};

struct TilesPlan {
    bool ok = false;
    TilesParams p{};
    int64_t group = 0;  // items run at a time
    int64_t words = 0;  // of scratch
    int64_t cblocks = 0;
    int32_t chans_per_block = 0;
    int cb = 1;         // channels of a point in LDS together
    int32_t bin_lds = 0, segment_lds = 0;  // bytes
};

constexpr int64_t kTilesFewGroups = 256;     // workgroups: one per CU
constexpr int64_t kTilesMost = 2048;         // per item: counts and masks of every tile in LDS (96 KiB)
constexpr int kTileBits = 11;
constexpr int64_t kTileBlocksMost = 2047;    // per item: segments of a tile in LDS (16 KiB), counts of 11 and 21 bits

constexpr int kCrowdedGroups = 1024;   // workgroups of that launch at most: with no tile on the list they cost it 2 us

template <int DIM>
inline TilesPlan tiles_plan_of(const GradGatherArgs& a)
{
    typedef GradTile<DIM> S;
    TilesPlan pl;
    if (a.interp > 1 || a.N < 1 || a.N > 65535 || a.W > INT32_MAX / 2 || a.H > INT32_MAX / 2 || a.D > INT32_MAX / 2) {
        return pl;
    }
    const int64_t esz = elem_size(a.elem);
    const int64_t tx = (a.W + S::kX - 1) / S::kX, ty = (a.H + S::kY - 1) / S::kY, tz = (a.D + S::kZ - 1) / S::kZ;
    if (tx > kTilesMost || ty > kTilesMost || tz > kTilesMost || tx * ty * tz > kTilesMost) {
        return pl;
    }
    const int64_t per_core = a.items_per_core > 0 ? a.items_per_core : 1;
    // the first block of an item starts at the boundary of the chunk that its first point lies in
    const int64_t blocks = (a.points + (per_core > 1 ? kBinPoints - 1 + 255 : kBinPoints - 1)) / kBinPoints;
    if (blocks > kTileBlocksMost) {
        return pl;
    }
    TilesParams& p = pl.p;
    p.C = (int32_t)a.C;
    p.D = (int32_t)a.D;
    p.H = (int32_t)a.H;
    p.W = (int32_t)a.W;
    p.points = (int32_t)a.points;
    p.pad = a.pad;
    p.align = a.align;
    p.items_per_core = (int32_t)per_core;
    p.elements = (int32_t)(a.D * a.H * a.W);
    p.tiles_x = (int32_t)tx;
    p.tiles_y = (int32_t)ty;
    p.tiles = (int32_t)(tx * ty * tz);
    p.blocks = (int32_t)blocks;
    // a point's corners lie in one tile or, with linear interpolation, in up to two along every axis
    p.lay.block_words = (uint32_t)(kBinPoints / 2) << (a.interp == 0 ? DIM : 0);
    p.lay.segments = 0;
    p.lay.records = align4((uint64_t)(blocks * p.tiles));
    p.lay.item_words = p.lay.records + (uint32_t)blocks * p.lay.block_words;
    const int64_t fit = kGatherGroupScratch / ((int64_t)p.lay.item_words * 4);
    const int64_t group = fit < 1 ? 1 : (fit < a.N ? fit : a.N);
    pl.group = (a.N + (a.N + group - 1) / group - 1) / ((a.N + group - 1) / group);  // as many items in every group
    p.N = (int32_t)pl.group;
    p.first_item = 0;
    p.crowded = crowded_tile(a);
    p.list_most = (uint32_t)(a.points > p.crowded.points || a.points > p.crowded.contributions ? pl.group * p.tiles : 0);
    p.list = (uint32_t)(pl.group * p.lay.item_words);
    pl.words = (int64_t)p.list + (p.list_most > 0 ? (int64_t)align4((uint64_t)p.list_most + 1u) : 0);
    pl.cb = (esz == 2 && a.C > 4 && DIM == 2) ? 8 : ((a.C > 3) ? 4 : (int)a.C);
    // fewer channels together where the tiles do not fill the chip
    while (pl.cb > 1 && pl.group * p.tiles * ((a.C + pl.cb - 1) / pl.cb) < kTilesFewGroups) {
        pl.cb = (pl.cb == 3) ? 2 : pl.cb / 2;
    }
    // channel blocks where the tiles alone do not fill the chip (four workgroups per CU): each makes the lists again
    const int64_t base = pl.group * p.tiles;
    const int64_t max_cblocks = (a.C + pl.cb - 1) / pl.cb;
    int64_t cblocks = (1024 + base - 1) / base;
    cblocks = cblocks > max_cblocks ? max_cblocks : cblocks;
    int64_t cpb = (a.C + cblocks - 1) / cblocks;
    cpb = (cpb + pl.cb - 1) / pl.cb * pl.cb;
    pl.cblocks = (a.C + cpb - 1) / cpb;
    pl.chans_per_block = (int32_t)cpb;
    p.by_tiles_x = make_fast_div((uint32_t)p.tiles_x);
    p.by_tiles_y = make_fast_div((uint32_t)p.tiles_y);
    p.by_tiles = make_fast_div((uint32_t)p.tiles);
    p.by_blocks = make_fast_div((uint32_t)p.blocks);
    p.by_item = make_fast_div((uint32_t)(p.tiles * pl.cblocks));
    pl.bin_lds = p.tiles * (kBinThreads / 64) * 12;
    pl.segment_lds = (p.blocks + 1) * 8;
    pl.ok = fits_launch(base * pl.cblocks + 8, S::kThreads) && fits_launch(pl.group * blocks + 8, kBinThreads);
    return pl;
}

// Whether the tiles are the faster way to sort (elsewhere the lists of gs_grad_gather_plan.hpp).  Input gradient alone, lists /
// tiles in microseconds, before there was a list of crowded tiles, which costs 4 to 7 where it is empty.
//
// As a rule they are: fp32 8x3x479x637 zeros 178 / 86, fp16 17x3x271x355 101 / 54, fp32 14x3x312x301 -> 388x374 nearest 245 / 96,
// fp16 1x14x236x198 -> 229x192 32 / 20, volumes bf16 13x5x27x47x57 108 / 86, fp32 10x2x14x26x17 nearest 24 / 15.
//
// Not in dense grids, where half of the elements have more contributions than keys and a tile takes several rounds: volumes
// from 1.25 points a voxel on (1x12x9x81x64 -> 13x117x93 130 / 237, 2x5x19x59x56 -> 27x85x80 169 / 211, 6x6x56x17x60 ->
// 65x19x70 134 / 164), planes from two an element on with many channels (21x60x40x40 -> 77x77 86 / 156; 10x2x267x440 ->
// 448x738 314 / 111) or border padding (14x4x33x56 -> 62x106 60 / 93), and bf16 coordinates beyond 64, whose eight bits gather
// points on whole and half pixels, from one on (2x5x96x192 -> 162x324 31 / 40, 12x5x100x129 -> 163x210 135 / 147; thinner ones
// 6x12x136x184 -> 115x156 47 / 34).
// Not where a single tile outlasts the launch: a workgroup adds the points that border padding piles up on a corner (a few in
// a hundred of an item) a thousand at a time, in lists a wavefront per element does, and with one or two items of many points
// and few channels nothing else is left to do meanwhile.  Which side is faster is the grid's doing; bilinear, both gradients, lists /
// tiles for rotations of up to 30 degrees (five grids), points at random, flow fields that stay inside:
//   1x3x384x552 -> 461x663        75 / 105  142 / 152   61 / 26     3x4x265x296                62 / 67    99 / 75    48 / 25
//   2x3x248x464                   80 / 83    98 / 80    46 / 22     fp16 5x3x232x296           76 / 76   110 / 78    50 / 28
//   2x4x578x571                  110 / 124  248 / 199  110 / 49     3x1x520x609 -> 605x708    198 / 180  282 / 213  123 / 66
//   fp16 1x6x180x170 (30600)      38 / 33    47 / 42    31 / 21     4x2x301x505               108 / 102  159 / 108   77 / 38
//   2x6x61x54                     34 / 24    36 / 21    29 / 15     5x2x405x480               176 / 137  219 / 150  113 / 57
// Over 182 calls of three to nine items tiles are 1.06, 1.37 and 1.64 times as fast, rotated ones slower in 64 (fp32 3x1x271x180 44 / 73
// at worst); over 13 of one and two items beyond 32768 points 0.89, 1.15 and 1.82, over 27 below 1.27, 1.32 and 1.50.  Nearest, which
// adds no weights, 1x2x368x624 47 / 39, 2x1x408x600 -> 792x1164 540 / 153, 3x2x304x576 144 / 77, 1x6x32x48 -> 44x66 20 / 20.
// Nor for many channels of volumes (12x31x18x62x20 142 / 159, 3x26x27x18x31 42 / 46; nearest 23x10x28x67x49 114 / 130,
// 5x28x9x71x45 35 / 39; 7x19x30x20x91 175 / 151, nearest 9x6x52x46x37 67 / 55).
// Not in planes and volumes of many tiles: every block of points clears, sums and writes a count per tile, and from 1706 tiles
// on a CU has room for one workgroup of that kernel.  fp32 4x3x720x1280 (1800 tiles) 158 / 220, reflection 168 / 269, nearest
// 113 / 166, 8x3x720x1280 323 / 428, 1x3x720x1280 58 / 66, 1x1x1024x1024 62 / 67, 4x3x1024x1024 -> 512x512 114 / 118; volumes
// 4x4x64x128x128 (2048) 300 / 461, 1x4 96 / 122.  One item of few points is faster by tiles: 1x1x1024x1024 -> 512x512 44 / 30.
// Below 1706, planes: one item 1x3x704x1152 (1584) 54 / 50, reflection (whose points lie closer at the edges) 60 / 62,
// 1x1x640x1120 (1400) 47 / 51; several 4x3x640x1120 125 / 129, nearest 90 / 101, reflection 133 / 157; 4x3x608x1024 (1216) 116 /
// 114, nearest 84 / 87, reflection 131 / 139; 4x3x600x800 (950) 99 / 77, reflection 107 / 99.  Volumes: 4x4x48x112x128 (1344) 198 /
// 173, reflection 272 / 242.
inline bool many_tiles(const GradGatherArgs& a)
{
    const int64_t elements = a.D * a.H * a.W;
    const int64_t tiles = a.dim == 3 ? ((a.W + 15) / 16) * ((a.H + 7) / 8) * ((a.D + 3) / 4) : ((a.W + 31) / 32) * ((a.H + 15) / 16);
    if (a.N == 1 && 2 * a.points <= elements) {
        return false;
    }
    const int64_t items = (a.dim == 2 && a.N > 1) ? 5 : 4, edges = (a.dim == 2 && a.pad == 2) ? 5 : 4;
    return tiles * items * edges > 1706 * 16;
}

inline bool tiles_are_faster(const GradGatherArgs& a)
{
    const int64_t elements = a.D * a.H * a.W;
    if (many_tiles(a)) {
        return false;
    }
    if (a.dim == 3) {
        return a.interp == 1 ? a.C <= 8 : (a.C <= 24 && 4 * a.points <= 5 * elements);
    }
    if (a.interp == 0 && a.points > 2 * elements && (a.C > 8 || a.pad == 1)) {
        return false;
    }
    if (a.interp == 0 && a.elem == Elem::BF16 && (a.H > 64 || a.W > 64) && a.points >= elements) {
        return false;
    }
    return a.pad != 1 || a.interp == 1 || a.N >= 3 || a.points <= 32768 || a.N * (a.C + 4) >= 48;
}

inline TilesPlan tiles_plan(const GradGatherArgs& a)
{
    if (!tiles_are_faster(a)) {
        return TilesPlan();
    }
    return a.dim == 3 ? tiles_plan_of<3>(a) : tiles_plan_of<2>(a);
}

}  // namespace opscv
