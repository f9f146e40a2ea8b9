// Backward of the grid samplers for gfx950: gradient of the input tile by tile, for planes and volumes, linear and
// nearest samples, any number of channels.
//
// The sum that reaches an element is a fixed sequence (gs2d_grad.hip, gs3d_grad.hip): its contributions ordered by
// (chunk of 256 grid points, tap, point), every add rounded to the element type.  Two kernels, no global atomics:
//
//   bin     a workgroup takes a block of 1024 consecutive grid points (whole chunks) and sorts them by the tile of the
//           plane that they contribute to, stably: every block leaves, per tile, a segment of 16-bit point numbers in
//           ascending order.  A point whose corners lie in several tiles is in the segments of all of them.
//   gather  a workgroup per tile, a lane per element: the tile's segments, block after block, are its points in
//           ascending order.  The points are counted by cell in LDS, every lane finds the runs of the cells that its
//           element is a corner of, keys them (chunk, tap, number in LDS), sorts the keys in registers and folds
//           weight times gradOutput, both from LDS, with the reference's roundings.  Elements with more contributions
//           than keys are merged, run by run, a lane each, or, where they are few or long, by the whole
//           wavefront; more points than LDS holds are taken a run of segments after the other, which are whole chunks
//           in ascending order.  Tiles that many points fall on are left to a third kernel (gs_grad_tiles_crowded.hip).
//
// The grid is read here and there, by the gather once per tile that a point reaches and block of channels, gradOutput once per
// tile that a point reaches; all that is scattered happens in LDS.
//
// fp32 8x3x479x637 from as many points (rotations of up to 30 degrees), operands from memory: lists through global memory
// (gs_grad_gather.hip) 188 us in six kernels, here bin 21, gather 71 and 4.5 for a list of crowded tiles that is empty (bin 19
// and gather 69 before there was one: where a point lies in its tile, and scalar registers that the way out takes).  With the gradient
// of the grid in its launch bin takes 53.5, 21 and 33 as two launches: they hardly overlap.  Bin: 34 us with an LDS atomic a point, which the
// 64 lanes of a wavefront on one tile take in turn, 20 with a run of lanes entered at once.  Gather is bound by its chain of
// steps, not by a unit: 550 vector, 400 scalar and 49 LDS instructions a wavefront (34 us of issue), and seven waits for memory
// or the other wavefronts (segments, records, points; counts, starts, lists, keys) at two workgroups per CU.  Without fetching,
// sorting and folding keys it takes 47 us, without gradOutput 63, without stores 64; three workgroups per CU (80 registers)
// are no faster, tiles of 32 x 8 take 92 us (and bin 61), half as many points a round 97.  Weights in LDS instead of
// coordinates took 82 to 80 us, loads of all of a lane's points together and divisions by multiplication 74, a reflection's
// constants out of the other paddings' way 69.  Volumes of four channels, linear, need more than the 128 registers that two
// workgroups per CU leave: 40 bytes of scratch a lane in fp32.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "gs_grad_gather.hpp"
#include "gs_grad_grid.hpp"
#include "gs_grad_points.hpp"
#include "gs_grad_tiles_kernel.hpp"
#include "gs_grad_tiles_plan.hpp"
#include "kernels.hpp"

namespace opscv {

namespace {

constexpr int kPosBits = 11;           // a point's number in LDS, or kRecords: none
constexpr int kTapBits = 3;
constexpr uint32_t kNoKey = 0xFFFFFFFFu;
constexpr uint32_t kNoPlace = 0xFFFFFFFFu;
// Runs of up to as many points are put in order by counting, longer ones by ballots.  32, 64 or 128: nearest, border padding,
// 1x1x704x912 73 / 70 / 69, 2x6x136x208 20 / 21 / 22 us; 79 and 22 with 32 and one read of LDS after the other.
constexpr uint32_t kCountedRun = 64;
// Crowded elements are put in order by a lane each where more than kFewCrowded lanes of a wavefront have one of up to kSerialMost
// contributions, otherwise one after the other by the wavefront, up to 64 * kRankedRegs contributions by counting.  A lane also
// adds up to kSerialMost by itself where more lanes than kFewCrowded have as many.  Longer ones are a lane each where the
// wavefront has kSideBySide times as many contributions as they: border padding piles points up on all elements of a row, and
// 32 of 88 contributions one after the other take the wavefront longer than a lane each (fp16 3x4x222x157 border, rotated 119 / 63
// us, 2x8x609x495 -> 649x527 377 / 178, volumes 6x13x17x11x45 -> 17x11x46 314 / 131; with 8 instead of 12 the elements of
// some hundred on a corner are a lane's too, fp32 5x2x167x179 78 for 53; with 24 3x6x286x208 remains at 131, 77 so;
// points at random close together lose, 11x10x246x80 -> 331x107 154 / 165).  Without the counting and with 192
// contributions / with it and 192 / 96 / 64 / 48 (and 16 lanes), microseconds of the whole gradient: fp32 reflection
// 5x4x27x54x51 81 / 66 / 67 / 67 / 66, fp16 3x3x31x45x16 50 / 41 / 41 / 39 / 49, fp32 9x22x25x16x29 86 / 66 / 66 / 67 / 74,
// planes, fp16 border 29x4x378x312 183 / 162 / 162 / 164 / 163; 22 such gradients together 1.10, 1.10, 1.10 and 1.05 times as
// fast, and 1.09 with 3 lanes instead of 6.
constexpr uint32_t kSerialMost = 64;
constexpr int kFewCrowded = 6;
constexpr uint32_t kSideBySide = 12;
constexpr int kRankedRegs = 2;

// What the bin kernel takes along: nothing, or the gradient of the grid by workgroups behind its own.
template <int DIM>
struct GridToo;
template <>
struct GridToo<2> {
    const void* gout;
    const void* x;
    void* dgrid;
    Grid2Params p;
};
template <>
struct GridToo<3> {
    const void* gout;
    const void* x;
    void* dgrid;
    Grid3Params p;
};

// the points of a workgroup of the grid's gradient
static_assert(kBinThreads == kGridTileThreads && kBinThreads == kChunkPoints3, "a lane a point in the bin kernel's workgroups");

// GRID: 0: no gradient of the grid; of planes 1 points in rows, 2 in tiles; of volumes 1 a channel's loads at a time, 2 four's
template <typename T, int DIM, int INTERP, int GRID>
__global__ __launch_bounds__(kBinThreads) void gs_tiles_bin_kernel(const T* __restrict__ grid, uint32_t* __restrict__ ws,
                                                                   TilesParams p, uint32_t pieces, uint32_t bin_blocks,
                                                                   GridToo<DIM> too)
{
    if constexpr (GRID != 0) {
        if (blockIdx.x >= bin_blocks) {
            const uint32_t block = blockIdx.x - bin_blocks;
            const T* gout = (const T*)too.gout;
            const T* x = (const T*)too.x;
            if constexpr (DIM == 2) {
                gs2d_grid_gradient_block<T, INTERP, GRID == 2>(block, gout, x, grid, (T*)too.dgrid, too.p);
            } else {
                gs3d_grid_gradient_block<T, INTERP, GRID == 2 ? 4 : 1>(block, gout, x, grid, (T*)too.dgrid, too.p);
            }
            return;
        }
    }
    typedef GradTile<DIM> S;
    constexpr int kWaves = kBinThreads / 64;
    constexpr int kSteps = kBinPoints / kBinThreads;
    constexpr int K = (INTERP == 0) ? (1 << DIM) : 1;  // tiles a point reaches at most
    extern __shared__ __align__(16) uint32_t smem[];
    __shared__ uint32_t s_total;
    uint32_t* counts = smem;                      // [wave][tile]
    unsigned long long* masks = reinterpret_cast<unsigned long long*>(smem + kWaves * p.tiles);  // [wave][tile]
    if (blockIdx.x == 0 && threadIdx.x == 0 && p.list_most > 0) {
        ws[p.list] = 0u;  // for the gather kernel
    }
    uint32_t n, block;
    if (!piece_of_block(blockIdx.x, pieces, p.by_blocks, &n, &block)) {
        return;
    }
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int32_t phase = (DIM == 3 && p.items_per_core > 1) ? phase_of(n, p) : 0;
    T raw[kSteps][DIM];  // all loads on their way before the first is looked at
    bool have[kSteps];
#pragma unroll
    for (int u = 0; u < kSteps; u++) {
        const int32_t pt = (int32_t)(block * kBinPoints) + wave * 256 + u * 64 + lane - phase;
        have[u] = pt >= 0 && pt < p.points;
        __builtin_memcpy(raw[u], grid + ((int64_t)n * p.points + (have[u] ? pt : 0)) * DIM, sizeof(raw[u]));
    }
    for (int i = t; i < kWaves * p.tiles * 3 / 4; i += kBinThreads) {
        reinterpret_cast<uint4*>(smem)[i] = make_uint4(0u, 0u, 0u, 0u);
    }
    if (t == 0) {
        s_total = 0u;
    }
    // The tiles of a point, -1 where it has no k-th one: that of its low corner, then those that the high corner lies in
    // along x, along y and so on; `any`: the k of which any lane of the wavefront has one.
    auto tiles_of = [&](int u, int32_t (&tile)[K], uint32_t (&part)[K], uint32_t* any) {
        int32_t x, y, z;
        const bool in = low_corner<T, DIM, INTERP>(coords_of<T, DIM, INTERP>(raw[u], p), p, &x, &y, &z) && have[u];
        auto low_of = [](int32_t v, int32_t edge) { return (int32_t)((uint32_t)(v < 0 ? 0 : v) / (uint32_t)edge); };
        auto next = [](int32_t v, int32_t size, int32_t edge) {  // the high corner lies in the next tile
            return v >= 0 && (v & (edge - 1)) == edge - 1 && v + 1 < size;
        };
        int32_t low = low_of(y, S::kY) * p.tiles_x + low_of(x, S::kX);
        if constexpr (DIM == 3) {
            low += low_of(z, S::kZ) * p.tiles_x * p.tiles_y;
        }
        const bool nx = next(x, p.W, S::kX), ny = next(y, p.H, S::kY), nz = DIM == 3 && next(z, p.D, S::kZ);
        // along an axis where it is the high corner that lies in the tile, that is in the first part
        uint32_t stride = 1;
        auto along = [&](int32_t v, int32_t edge, int32_t part_edge, int axis) {
            const uint32_t in_tile = (uint32_t)(v < 0 ? 0 : v) & (uint32_t)(edge - 1);
            const bool spills = INTERP == 0 && v >= 0 && (in_tile & (uint32_t)(part_edge - 1)) == (uint32_t)(part_edge - 1) &&
                                in_tile != (uint32_t)(edge - 1);
            const uint32_t code = in_tile / (uint32_t)part_edge * stride | (spills ? 1u << (kRecordPartBits + axis) : 0u);
            stride *= (uint32_t)(edge / part_edge);
            return code;
        };
        const uint32_t part_x = along(x, S::kX, S::kPartX, 0), part_y = along(y, S::kY, S::kPartY, 1);
        const uint32_t part_z = (DIM == 3) ? along(z, S::kZ, S::kPartZ, 2) : 0u;
        *any = 1u;
#pragma unroll
        for (int k = 0; k < K; k++) {
            const bool is = in && (!(k & 1) || nx) && (!(k & 2) || ny) && (!(k & 4) || nz);
            tile[k] = is ? low + (k & 1) + ((k & 2) ? p.tiles_x : 0) + ((k & 4) ? p.tiles_x * p.tiles_y : 0) : -1;
            part[k] = ((k & 1) ? 0u : part_x) + ((k & 2) ? 0u : part_y) + ((k & 4) ? 0u : part_z);
            if (k > 0) {
                *any |= __builtin_amdgcn_ballot_w64(is) != 0 ? 1u << k : 0u;
            }
        }
    };
    // The rank of a point among those of its tile in earlier lanes and steps of the wavefront, from a mask of the tile's
    // lanes.  Neighbouring points share tiles: the first of a run of lanes with one tile enters the whole run (an atomic of
    // 64 lanes on one address would take 64 turns).
    uint32_t* mine = counts + wave * p.tiles;
    unsigned long long* my_masks = masks + wave * p.tiles;
    uint32_t place[kSteps][K], any[kSteps];  // part << 20 | tile << 8 | rank among the wavefront's 256 points
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kSteps; u++) {
        int32_t tile[K];
        uint32_t part[K];
        tiles_of(u, tile, part, &any[u]);
#pragma unroll
        for (int k = 0; k < K; k++) {
            place[u][k] = kNoPlace;
            if ((any[u] >> k) & 1u) {
                const int32_t left = __builtin_amdgcn_update_dpp(-2, tile[k], 0x138, 0xf, 0xf, false);  // of the lane before
                const bool begins = left != tile[k];
                const uint64_t bounds = __builtin_amdgcn_ballot_w64(begins);
                if (begins && tile[k] >= 0) {
                    const uint64_t from_here = ~0ull << lane, later = bounds & (from_here << 1);
                    atomicOr(&my_masks[tile[k]], (unsigned long long)(((later & (0ull - later)) - 1ull) & from_here));
                }
            }
        }
        landed();
        uint64_t mask[K];
        uint32_t before[K];
#pragma unroll
        for (int k = 0; k < K; k++) {
            if (((any[u] >> k) & 1u) && tile[k] >= 0) {
                mask[k] = my_masks[tile[k]];
                before[k] = mine[tile[k]];
            }
        }
        landed();
#pragma unroll
        for (int k = 0; k < K; k++) {
            if (((any[u] >> k) & 1u) && tile[k] >= 0) {
                const uint32_t below = bits_below(mask[k]);
                place[u][k] = (part[k] << 20) | ((uint32_t)tile[k] << 8) | (before[k] + below);
                if (below == 0u) {
                    mine[tile[k]] = before[k] + (uint32_t)__builtin_popcountll(mask[k]);
                    my_masks[tile[k]] = 0ull;
                }
            }
        }
        landed();
    }
    __syncthreads();
    // a run of the block's records per tile (the order of the runs does not matter), and within it one per wavefront
    uint32_t* wsn = ws + (size_t)n * p.lay.item_words;
    for (int32_t i0 = 0; i0 < p.tiles; i0 += kBinThreads) {
        const int32_t i = i0 + t;
        uint32_t of[kWaves], sum = 0;
#pragma unroll
        for (int w = 0; w < kWaves; w++) {
            of[w] = (i < p.tiles) ? counts[w * p.tiles + i] : 0u;
            sum += of[w];
        }
        uint32_t start = 0;
        if (__builtin_amdgcn_ballot_w64(sum != 0u) != 0) {
            const uint32_t incl = wave_scan(sum);
            uint32_t base = 0;
            if (lane == 63) {
                base = atomicAdd(&s_total, incl);
            }
            start = (uint32_t)__builtin_amdgcn_readlane((int)base, 63) + incl - sum;
            if (sum != 0u) {
                uint32_t begin = start;
#pragma unroll
                for (int w = 0; w < kWaves; w++) {
                    counts[w * p.tiles + i] = begin;
                    begin += of[w];
                }
            }
        }
        if (i < p.tiles) {
            wsn[p.lay.segments + (size_t)block * p.tiles + i] = start | (sum << 16);
        }
    }
    __syncthreads();
    uint16_t* records = reinterpret_cast<uint16_t*>(wsn + p.lay.records + (size_t)block * p.lay.block_words);
#pragma unroll
    for (int u = 0; u < kSteps; u++) {
#pragma unroll
        for (int k = 0; k < K; k++) {
            if (((any[u] >> k) & 1u) && place[u][k] != kNoPlace) {
                const uint32_t at = mine[(place[u][k] >> 8) & 0xFFFu] + (place[u][k] & 255u);
                records[at] = (uint16_t)((place[u][k] >> 20 << kRecordBits) | (uint32_t)(wave * 256 + u * 64 + lane));
            }
        }
    }
}

// Ascending, by Batcher's odd-even merge sort (cut to N keys: the ones past the end would stay there): 12 comparators for
// 6 keys, 19 for 8, 41 for 12, 63 for 16, 127 for 24.
template <int N>
__device__ __forceinline__ void sort_keys(uint32_t* key)
{
#pragma unroll
    for (int p = 1; p < N; p *= 2) {
#pragma unroll
        for (int k = p; k >= 1; k /= 2) {
#pragma unroll
            for (int j = k % p; j + k < N; j += 2 * k) {
#pragma unroll
                for (int i = 0; i < k; i++) {
                    const int l = i + j, h = i + j + k;
                    if (h < N && l / (2 * p) == h / (2 * p)) {
                        const uint32_t a = key[l], b = key[h];
                        key[l] = a < b ? a : b;
                        key[h] = a < b ? b : a;
                    }
                }
            }
        }
    }
}

// The network for `most` keys, a multiple of STEP up to N.
template <int N, int STEP>
__device__ __forceinline__ void sort_most(uint32_t* key, int most)
{
    if (most == N) {
        sort_keys<N>(key);
    } else if constexpr (N > STEP) {
        sort_most<N - STEP, STEP>(key, most);
    }
}

// The sums of an element's channels.  A contribution is weight times gradOutput rounded to the element type, added with a
// rounding to the element type.  For fp16 both steps are the native instructions, two channels at a time: the product of
// two fp16 values is exact in fp32, so rounding it to fp16 is the fp16 product, and the fp32 sum of two fp16 values rounded
// to fp16 is the fp16 sum (24 >= 2 x 11 + 2 bits).
template <typename T, int INTERP, int CB>
struct Sums {
    float v[CB];
    __device__ __forceinline__ void clear()
    {
#pragma unroll
        for (int j = 0; j < CB; j++) {
            v[j] = 0.0f;
        }
    }
    __device__ __forceinline__ void add(const T* go, float w)
    {
#pragma unroll
        for (int j = 0; j < CB; j++) {
            v[j] = rt<T>(v[j] + value_of<T, INTERP>(ElemIO<T>::load(go + j), w));
        }
    }
    __device__ __forceinline__ float get(int j) const { return v[j]; }
    __device__ __forceinline__ void set(int j, float f) { v[j] = f; }
};
template <int INTERP, int CB>
struct Sums<_Float16, INTERP, CB> {
    typedef _Float16 pair_t __attribute__((ext_vector_type(2)));
    static constexpr int P = (CB + 1) / 2;
    pair_t v[P];
    __device__ __forceinline__ void clear()
    {
#pragma unroll
        for (int j = 0; j < P; j++) {
            v[j] = (pair_t)((_Float16)0.0f);
        }
    }
    __device__ __forceinline__ void add(const _Float16* go, float w)
    {
        const pair_t ww = (pair_t)((_Float16)w);  // exact
#pragma unroll
        for (int j = 0; j < P; j++) {
            pair_t g;
            g.x = go[2 * j];
            g.y = (2 * j + 1 < CB) ? go[(2 * j + 1 < CB) ? 2 * j + 1 : 0] : (_Float16)0.0f;
            const pair_t val = (INTERP == 1) ? g : g * ww;
            v[j] = v[j] + val;
        }
    }
    __device__ __forceinline__ float get(int j) const { return (float)((j & 1) ? v[j >> 1].y : v[j >> 1].x); }
    __device__ __forceinline__ void set(int j, float f)
    {
        if (j & 1) {
            v[j >> 1].y = (_Float16)f;
        } else {
            v[j >> 1].x = (_Float16)f;
        }
    }
};

template <typename T, int DIM, int INTERP, int CB>
__global__ __launch_bounds__(GradTile<DIM>::kThreads, 4) void gs_tiles_gather_kernel(
    const T* __restrict__ gout, const T* __restrict__ grid, T* __restrict__ dx, const uint32_t* __restrict__ ws,
    uint32_t* __restrict__ list, TilesParams p, uint32_t pieces, int32_t chans_per_block)
{
    typedef GradTile<DIM> S;
    constexpr int TH = S::kThreads, CAP = S::kRecords, RPL = (CAP + TH - 1) / TH, kWaves = TH / 64;
    static_assert(CAP % 64 == 0 && CAP >= kBinPoints && CAP < (1 << kPosBits), "whole segments, numbers that fit a key");
    static_assert(DIM == 3 || S::kX * kWaves * (64 / S::kX) == TH, "whole rows in a wavefront");
    static_assert(kWaves <= 16, "totals of the wavefronts in a row of lanes");
    constexpr int PADC = (INTERP == 0) ? 1 : 0;  // cells beside the first element of a row
    constexpr int CX = S::kX + PADC, CY = S::kY + PADC, CZ = (DIM == 3) ? S::kZ + PADC : 1;
    constexpr int CELLS = CX * CY * CZ;
    constexpr int RR = (INTERP == 0) ? (1 << (DIM - 1)) : 1;  // rows of cells: a row's two cells are neighbours in the list
    constexpr int R = (INTERP == 0) ? 2 * RR : 1;             // runs
    constexpr int GS = (CB == 3) ? 4 : CB;                    // of a point's gradOutput in LDS
    constexpr int NK = (DIM == 3 && INTERP == 0) ? 24 : 16;   // keys of an element, in steps of
    constexpr int kStep = (DIM == 3 && INTERP == 0) ? 4 : 2;
    constexpr int kStarts = (CELLS + 1 + 3) / 4 * 4;
    // a point of a plane is a contribution of four elements: all crowded ones fit; of volumes most do
    constexpr uint32_t kSorted = (INTERP == 1) ? CAP : ((DIM == 3) ? 3072 : 4 * CAP);
    constexpr uint32_t kLowBits = (1u << (kPosBits + kTapBits)) - 1u;
    __shared__ __align__(16) uint32_t s_start[kStarts];  // counts by cell, then the start of every cell's run in s_list
    __shared__ uint32_t s_list[CAP + 2 * NK];  // keys by cell; lanes read past the end of their runs
    __shared__ Weights<T, DIM, (INTERP == 0) ? CAP : 0> s_weight;
    __shared__ __align__(16) T s_go[(CAP + 1) * GS];  // the last: zeros
    // of crowded elements: while lists are put in order, then while contributions are added
    struct ByPoint {
        uint32_t key[CAP];  // chunk, parity of the cell along every axis, the point's number: ascending
        uint16_t cell[CAP];
    };
    struct ByWave {
        float value[CB][68];
        uint16_t order[64];
    };
    union Rare {
        ByPoint points;
        ByWave waves[kWaves];
    };
    __shared__ __align__(16) Rare s_rare;
    __shared__ uint16_t s_long[CAP / kCountedRun + 1];
    __shared__ uint32_t s_scan[kWaves];
    __shared__ uint16_t s_sorted[kSorted];  // contributions of crowded elements in order: the low bits of their keys
    __shared__ uint32_t s_longs, s_crowded, s_sorted_used;
    extern __shared__ uint32_t s_seg[];  // per segment that is not empty: points before it; block << 14 | first record
    uint32_t n, local;
    if (!piece_of_block(blockIdx.x, pieces, p.by_item, &n, &local)) {
        return;
    }
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t cblock = fast_div(local, p.by_tiles), tile = local - cblock * (uint32_t)p.tiles;
    const uint32_t* wsn = ws + (size_t)n * p.lay.item_words;
    const uint16_t* records = reinterpret_cast<const uint16_t*>(wsn + p.lay.records);
    const int32_t tile_yz = (int32_t)fast_div(tile, p.by_tiles_x), tile_x = (int32_t)tile - tile_yz * p.tiles_x;
    const int32_t tile_z = (DIM == 3) ? (int32_t)fast_div((uint32_t)tile_yz, p.by_tiles_y) : 0;
    const int32_t tile_y = tile_yz - tile_z * p.tiles_y;
    const int32_t x0 = tile_x * S::kX, y0 = tile_y * S::kY, z0 = tile_z * S::kZ;
    const int32_t phase = (DIM == 3 && p.items_per_core > 1) ? phase_of(n, p) : 0;
    auto wave_sum = [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane((int)wave_scan(v), 63); };
    auto waves_before = [&](uint32_t* all) { return sums_before<kWaves>(s_scan, wave, lane, all); };

    uint32_t* s_before = s_seg;
    uint32_t* s_where = s_seg + p.blocks + 1;
    uint32_t segs, total;
    tile_segments<TH>(wsn, p, tile, s_before, s_where, s_scan, &segs, &total);
    // to gs_tiles_crowded_kernel; every tile has room on the list.  One number is all that is kept for it: scalar registers are
    // what this kernel has too few of
    const uint32_t entry = cblock == 0u ? (n << kTileBits) | tile : kNoPlace;
    auto leave = [&]() {
        if (entry != kNoPlace && t == 0) {
            list[1u + atomicAdd(list, 1u)] = entry;
        }
    };
    if (total > p.crowded.points) {
        leave();
        return;
    }
    if (t < GS) {
        ElemIO<T>::store(&s_go[CAP * GS + t], 0.0f);
    }
    if (INTERP == 0) {
        s_weight.clear_last(t);
    }
    for (int i = t; i < CAP + 2 * NK; i += TH) {
        s_list[i] = 0u;
    }
    __syncthreads();

    // rows of a plane to different wavefronts in turn: neighbours on which padding piles points up are then summed side by side
    const int row = (DIM == 2) ? wave + (lane / S::kX) * kWaves : t / S::kX;
    const int lx = t % S::kX, ly = row % S::kY, lz = row / S::kY;
    const int32_t c_begin = (int32_t)cblock * chans_per_block;
    const int32_t c_end = (c_begin + chans_per_block < p.C) ? c_begin + chans_per_block : p.C;
    const T* go_n = gout + (int64_t)n * p.C * (int64_t)p.points;
    const T* grid_n = grid + (int64_t)n * p.points * DIM;

    int32_t pt[RPL];                // the lane's points of this run of segments
    uint32_t key[NK];
    uint32_t len = 0, number = 0;   // contributions; points in LDS
    int most = 0;                   // keys of any lane of the wavefront
    bool crowded = false;
    uint32_t sorted = kNoKey;       // where a crowded element's contributions lie in s_sorted, or
    uint32_t only = kNoKey;         // in s_list: those of a single run
    // which corner of the element's cells a point is follows from the parity of its cell: 1 for the cell before
    const uint32_t parity = (INTERP == 1) ? 0u
                                          : (uint32_t)((lx & 1) | ((ly & 1) << 1) | ((DIM == 3) ? (lz & 1) << 2 : 0)) << kPosBits;
    constexpr uint32_t kCorners = (INTERP == 1) ? 0u : ((1u << DIM) - 1u) << kPosBits;
    const uint32_t corner = parity ^ kCorners;
    // the first cell of a row of an element's cells
    auto row_of = [&](int r) {
        if (INTERP == 1) {
            return (uint32_t)((lz * CY + ly) * CX + lx);
        }
        const int ys = r & 1, zs = r >> 1;
        return (uint32_t)((((DIM == 3) ? (lz + 1 - zs) * CY : 0) + ly + 1 - ys) * CX + lx);
    };
    constexpr uint32_t kRowCells = (INTERP == 1) ? 1u : 2u;

    auto lane_points = [&](int k) { return (uint32_t)(k * TH + wave * 64) < number; };  // any in this wavefront
    auto load_go = [&](int32_t c0, int32_t nc, int k, T (&go)[GS]) {
        const char* base = reinterpret_cast<const char*>(go_n + (int64_t)c0 * p.points);
        const uint32_t off = (uint32_t)pt[k] * (uint32_t)sizeof(T);  // an item's grid points fit 32 bits many times over
        auto load = [&](int j) {
            return *reinterpret_cast<const T*>(base + (int64_t)j * p.points * (int64_t)sizeof(T) + off);
        };
        if (nc == CB) {
#pragma unroll
            for (int j = 0; j < CB; j++) {
                go[j] = load(j);
            }
        } else {
#pragma unroll
            for (int j = 0; j < CB; j++) {
                go[j] = load(j < nc ? j : 0);
            }
        }
        if (GS > CB) {
            ElemIO<T>::store(&go[GS - 1], 0.0f);
        }
    };
    auto stage_go = [&](int k, const T (&go)[GS]) {
        const uint32_t i = (uint32_t)(k * TH + t);
        if (i < number) {
            __builtin_memcpy(__builtin_assume_aligned(&s_go[i * GS], sizeof(T) * GS), go, sizeof(T) * GS);
        }
    };

    // run r of the list: the points that corner r of this element comes from
    auto runs_of_element = [&](uint32_t (&begin)[R], uint32_t (&end)[R]) {
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint32_t cell = row_of(r >> 1) + ((INTERP == 1 || (r & 1)) ? 0u : 1u);
            begin[r] = s_start[cell];
            end[r] = s_start[cell + 1u];
        }
    };
    // f(key) for the contributions of a lane's element in order: the least of its runs' next keys
    auto merge_alone = [&](auto&& f) {
        uint32_t at[R], end[R], head[R];
        runs_of_element(at, end);
        auto next = [&](int r) { return (at[r] < end[r]) ? s_list[at[r]] ^ corner : kNoKey; };
#pragma unroll
        for (int r = 0; r < R; r++) {
            head[r] = next(r);
        }
        for (uint32_t i = 0; i < len; i++) {
            uint32_t least = head[0];
#pragma unroll
            for (int r = 1; r < R; r++) {
                least = head[r] < least ? head[r] : least;
            }
            f(i, least);
#pragma unroll
            for (int r = 0; r < R; r++) {
                if (head[r] == least) {
                    at[r]++;
                    head[r] = next(r);
                }
            }
        }
    };
    // the contributions of lane `owner`'s element by the whole wavefront: the least 64 of its runs' next 64 each are put(place
    // among them, key), then done(how many)
    auto merge_together = [&](int owner, int lane, auto&& put, auto&& done) {
        uint32_t begin[R], left[R], rest = 0;
        runs_of_element(begin, left);
#pragma unroll
        for (int r = 0; r < R; r++) {
            begin[r] = (uint32_t)__builtin_amdgcn_readlane((int)begin[r], owner);
            left[r] = (uint32_t)__builtin_amdgcn_readlane((int)left[r], owner) - begin[r];
            rest += left[r];
        }
        const uint32_t its_corner = (uint32_t)__builtin_amdgcn_readlane((int)corner, owner);
        while (rest > 0u) {
            const uint32_t batch = rest < 64u ? rest : 64u;
            uint32_t head[R], window[R];
#pragma unroll
            for (int r = 0; r < R; r++) {
                window[r] = left[r] < 64u ? left[r] : 64u;
                head[r] = ((uint32_t)lane < window[r]) ? s_list[begin[r] + lane] ^ its_corner : kNoKey;
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                uint32_t rank = (uint32_t)lane;
#pragma unroll
                for (int o = 0; o < R; o++) {
                    if (o != r && window[o] > 0u && window[r] > 0u) {
                        // keys of run o below this lane's
                        uint32_t less = 0;
#pragma unroll
                        for (uint32_t d = 32; d > 0u; d >>= 1) {
                            const uint32_t other = (uint32_t)__shfl((int)head[o], (int)(less + d - 1u));
                            less += (other < head[r]) ? d : 0u;
                        }
                        // the last of 64
                        less += ((uint32_t)__shfl((int)head[o], (int)less) < head[r]) ? 1u : 0u;
                        rank += less;
                    }
                }
                const bool take = (uint32_t)lane < window[r] && rank < batch;
                if (take) {
                    put(rank, head[r] & kLowBits);
                }
                const uint32_t taken = (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(take));
                begin[r] += taken;
                left[r] -= taken;
            }
            rest -= batch;
            done(batch);
        }
    };
    // The same for up to 64 * kRankedRegs contributions: a key or some a lane, whose place is the number of lesser ones.  (By
    // itself a lane waits for LDS at every contribution, some 200 clocks; here a contribution costs 10.)
    auto rank_together = [&](int owner, int lane, uint32_t its_len, auto&& put) {
        uint32_t first[R], end[R];  // of the runs: where their keys lie in the list, less those of the runs before; sums
        runs_of_element(first, end);
        uint32_t sum = 0;
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint32_t begin = (uint32_t)__builtin_amdgcn_readlane((int)first[r], owner);
            const uint32_t upto = (uint32_t)__builtin_amdgcn_readlane((int)end[r], owner);
            first[r] = begin - sum;
            sum += upto - begin;
            end[r] = sum;
        }
        const uint32_t its_corner = (uint32_t)__builtin_amdgcn_readlane((int)corner, owner);
        uint32_t own[kRankedRegs], rank[kRankedRegs];
#pragma unroll
        for (int m = 0; m < kRankedRegs; m++) {
            const uint32_t i = (uint32_t)(m * 64 + lane);
            uint32_t from = first[0];
#pragma unroll
            for (int r = 1; r < R; r++) {
                from = i >= end[r - 1] ? first[r] : from;
            }
            own[m] = (i < its_len) ? s_list[from + i] ^ its_corner : kNoKey;
            rank[m] = 0u;
        }
#pragma unroll
        for (int m = 0; m < kRankedRegs; m++) {
            const uint32_t n_keys = its_len > (uint32_t)(m * 64) ? its_len - (uint32_t)(m * 64) : 0u;
            const uint32_t here = n_keys < 64u ? n_keys : 64u;
            for (uint32_t j = 0; j < here; j += 8u) {
#pragma unroll
                for (uint32_t u = 0; u < 8u; u++) {
                    const uint32_t other = (uint32_t)__builtin_amdgcn_readlane((int)own[m], (int)(j + u));
#pragma unroll
                    for (int q = 0; q < kRankedRegs; q++) {
                        rank[q] += (other < own[q]) ? 1u : 0u;
                    }
                }
            }
        }
#pragma unroll
        for (int m = 0; m < kRankedRegs; m++) {
            if ((uint32_t)(m * 64 + lane) < its_len) {
                put(rank[m], own[m] & kLowBits);
            }
        }
    };
    // The contributions of crowded elements in order to s_sorted, once for all channels: a lane each, or where a single
    // element has hundreds the wavefront together.
    auto merge_crowded = [&]() {
        sorted = kNoKey;
        if (__builtin_amdgcn_ballot_w64(crowded) == 0) {
            return;
        }
        bool fits = false;
        if (crowded) {
            uint32_t begin[R], end[R];
            runs_of_element(begin, end);
            only = kNoKey;
#pragma unroll
            for (int r = 0; r < R; r++) {
                only = (end[r] - begin[r] == len) ? begin[r] : only;
            }
            if (only == kNoKey) {
                const uint32_t to = atomicAdd(&s_sorted_used, len);
                fits = to + len <= kSorted;
                sorted = fits ? to : kNoKey;
            }
        }
        const bool few = __builtin_popcountll(__builtin_amdgcn_ballot_w64(fits)) <= kFewCrowded;
        const uint32_t all = wave_sum(fits ? len : 0u);
        const bool alone = fits && ((!few && len <= kSerialMost) || len * kSideBySide <= all);
        if (alone) {
            merge_alone([&](uint32_t i, uint32_t k) { s_sorted[sorted + i] = (uint16_t)(k & kLowBits); });
        }
        int lane = t & 63;
        asm volatile("" : "+v"(lane));  // what follows is rare: none of it is worked out ahead
        uint64_t big = __builtin_amdgcn_ballot_w64(fits && !alone);
        while (big != 0) {
            const int owner = __builtin_ctzll(big);
            big &= big - 1u;
            uint32_t to = (uint32_t)__builtin_amdgcn_readlane((int)sorted, owner);
            const uint32_t its_len = (uint32_t)__builtin_amdgcn_readlane((int)len, owner);
            if (its_len <= 64u * kRankedRegs) {
                rank_together(owner, lane, its_len, [&](uint32_t rank, uint32_t k) { s_sorted[to + rank] = (uint16_t)k; });
                continue;
            }
            merge_together(owner, lane, [&](uint32_t rank, uint32_t k) { s_sorted[to + rank] = (uint16_t)k; },
                           [&](uint32_t batch) { to += batch; });
        }
        landed();
    };

    // the points of segments [from, to): cells, lists, and this element's keys in order; whether the tile is another kernel's
    auto build = [&](uint32_t from, uint32_t to, int32_t c0, int32_t nc) {
        const uint32_t base = s_before[from];
        number = s_before[to] - base;
        for (int i = t; i < kStarts / 4; i += TH) {
            reinterpret_cast<uint4*>(s_start)[i] = make_uint4(0u, 0u, 0u, 0u);
        }
        if (t == 0) {
            s_longs = s_crowded = s_sorted_used = 0u;
        }
        uint32_t own_key[RPL], rank[RPL], cell[RPL];
        T raw[RPL][DIM], go[RPL][GS];
        // stage by stage for all of the lane's points, so that their loads are on their way together
        uint32_t steps = 1;
        while (steps < to - from) {
            steps <<= 1;
        }
        uint32_t block[RPL];
        uint16_t record[RPL];
#pragma unroll
        for (int k = 0; k < RPL; k++) {
            if (lane_points(k)) {
                uint32_t i = (uint32_t)(k * TH + t);
                i = base + (i < number ? i : 0u);
                uint32_t seg = from;  // the last segment that does not start behind point i
                for (uint32_t d = steps >> 1; d > 0u; d >>= 1) {
                    const uint32_t mid = seg + d < to ? seg + d : to;
                    seg = s_before[mid] <= i ? mid : seg;
                }
                const uint32_t where = s_where[seg];
                block[k] = where >> 14;
                record[k] = *reinterpret_cast<const uint16_t*>(
                    reinterpret_cast<const char*>(records) +
                    (block[k] * (p.lay.block_words * 4u) + ((where & 0x3FFFu) + (i - s_before[seg])) * 2u));
            }
        }
#pragma unroll
        for (int k = 0; k < RPL; k++) {
            if (lane_points(k)) {
                const uint32_t q = block[k] * kBinPoints + (record[k] & (kBinPoints - 1u));
                pt[k] = (int32_t)q - phase;
                own_key[k] = (q >> 8) << (kPosBits + kTapBits);
                __builtin_memcpy(raw[k], reinterpret_cast<const char*>(grid_n) + (uint32_t)pt[k] * (uint32_t)sizeof(raw[k]), sizeof(raw[k]));
                load_go(c0, nc, k, go[k]);
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < RPL; k++) {
            if (lane_points(k)) {
                const uint32_t i = (uint32_t)(k * TH + t);
                const Coords<T, DIM> at = coords_of<T, DIM, INTERP>(raw[k], p);
                int32_t cx, cy, cz;
                low_corner<T, DIM, INTERP>(at, p, &cx, &cy, &cz);
                cx += PADC - x0;
                cy += PADC - y0;
                cz += PADC - z0;
                cell[k] = (uint32_t)((((DIM == 3) ? cz * CY : 0) + cy) * CX + cx);
                cell[k] = cell[k] < (uint32_t)CELLS ? cell[k] : 0u;  // never: the point is in this tile's segment
                const uint32_t odd = (uint32_t)((cx & 1) | ((cy & 1) << 1) | ((DIM == 3) ? (cz & 1) << 2 : 0)) << kPosBits;
                own_key[k] |= (INTERP == 1 ? 0u : odd) | i;
                rank[k] = 0u;
                if (i < number) {
                    rank[k] = atomicAdd(&s_start[cell[k]], 1u);
                    s_rare.points.key[i] = own_key[k];
                    s_rare.points.cell[i] = (uint16_t)cell[k];
                    if constexpr (INTERP == 0) {
                        s_weight.put(i, at);
                    }
                }
                stage_go(k, go[k]);
            }
        }
        __syncthreads();
        // the starts: four cells a lane
        uint4 four = make_uint4(0u, 0u, 0u, 0u);
        uint32_t incl = 0, sum = 0;
        if (t < kStarts / 4) {
            four = reinterpret_cast<uint4*>(s_start)[t];
        }
        if (wave * 64 < kStarts / 4) {
            sum = four.x + four.y + four.z + four.w;
            incl = wave_scan(sum);
        }
        if (lane == 63) {
            s_scan[wave] = incl;
        }
        __syncthreads();
        if (wave * 64 < kStarts / 4) {
            uint32_t all;
            const uint32_t before = waves_before(&all) + incl - sum;
            if (t < kStarts / 4) {
                reinterpret_cast<uint4*>(s_start)[t] =
                    make_uint4(before, before + four.x, before + four.x + four.y, before + four.x + four.y + four.z);
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < RPL; k++) {
            if ((uint32_t)(k * TH + t) < number) {
                s_list[s_start[cell[k]] + rank[k]] = own_key[k];
            }
        }
        uint32_t from_row[RR], upto[RR];  // where the row's keys lie in the list, less those of the rows before; contributions
        len = 0u;
#pragma unroll
        for (int r = 0; r < RR; r++) {
            const uint32_t row = row_of(r), begin = s_start[row];
            from_row[r] = begin - len;
            len += s_start[row + kRowCells] - begin;
            upto[r] = len;
        }
        len = (x0 + lx < p.W && y0 + ly < p.H && z0 + lz < p.D) ? len : 0u;
        crowded = len > (uint32_t)NK;
        if (crowded) {
            atomicOr(&s_crowded, len > p.crowded.contributions ? 3u : 1u);
        }
        __syncthreads();
        if (s_crowded != 0u) {
            if (INTERP == 0 && from == 0u && s_crowded == 3u) {
                return true;
            }
            // merging wants the points of a cell in order
            uint32_t place[RPL];
#pragma unroll
            for (int k = 0; k < RPL; k++) {
                const uint32_t i = (uint32_t)(k * TH + t);
                place[k] = 0xFFFFu;
                if (i < number) {
                    const uint32_t begin = s_start[cell[k]], end = s_start[cell[k] + 1u];
                    if (end - begin <= kCountedRun) {
                        uint32_t less = 0;
                        for (uint32_t j = begin; j < end; j += 4u) {  // of one cell: in the order of their numbers
                            uint32_t other[4];
#pragma unroll
                            for (uint32_t u = 0; u < 4u; u++) {
                                other[u] = s_list[j + u < end ? j + u : begin];
                            }
#pragma unroll
                            for (uint32_t u = 0; u < 4u; u++) {
                                less += (j + u < end && other[u] < own_key[k]) ? 1u : 0u;
                            }
                        }
                        place[k] = begin + less;
                    } else if (rank[k] == 0u) {
                        s_long[atomicAdd(&s_longs, 1u)] = (uint16_t)cell[k];
                    }
                }
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < RPL; k++) {
                if (place[k] != 0xFFFFu) {
                    s_list[place[k]] = own_key[k];
                }
            }
            for (uint32_t r = (uint32_t)wave; r < s_longs; r += kWaves) {
                const uint32_t c = s_long[r];
                uint32_t to_list = s_start[c];
                for (uint32_t i0 = 0; i0 < number; i0 += 256u) {
                    uint32_t its_cell[4], key[4];
#pragma unroll
                    for (uint32_t u = 0; u < 4u; u++) {
                        const uint32_t i = i0 + u * 64u + (uint32_t)lane;
                        its_cell[u] = s_rare.points.cell[i < number ? i : 0u];
                        key[u] = s_rare.points.key[i < number ? i : 0u];
                    }
#pragma unroll
                    for (uint32_t u = 0; u < 4u; u++) {
                        const bool member = i0 + u * 64u + (uint32_t)lane < number && its_cell[u] == c;
                        const uint64_t mask = __builtin_amdgcn_ballot_w64(member);
                        if (member) {
                            s_list[to_list + bits_below(mask)] = key[u];
                        }
                        to_list += (uint32_t)__builtin_popcountll(mask);
                    }
                }
            }
            __syncthreads();
            merge_crowded();
        }
        // Keys of as many contributions as any lane of the wavefront has, rounded up to kStep: beyond its own a lane reads
        // some key of the list and takes that of the zeros instead.
        const uint32_t keys = crowded ? 0u : len;
        most = 0;
#pragma unroll
        for (int i = 0; i < NK; i += kStep) {
            most = (__builtin_amdgcn_ballot_w64(keys > (uint32_t)i) != 0) ? i + kStep : most;
        }
#pragma unroll
        for (int r = 0; r < RR; r++) {
            from_row[r] = crowded ? 0u : from_row[r];
        }
#pragma unroll
        for (int g = 0; g < NK; g += kStep) {
            if (g < most) {
#pragma unroll
                for (int i = g; i < g + kStep; i++) {
                    uint32_t row = from_row[0];
#pragma unroll
                    for (int r = 1; r < RR; r++) {
                        row = ((uint32_t)i >= upto[r - 1]) ? from_row[r] : row;
                    }
                    const uint32_t k = s_list[row + (uint32_t)i] ^ corner;
                    key[i] = ((uint32_t)i < keys) ? k : (kNoKey << kPosBits) | (uint32_t)CAP;
                }
            }
        }
        sort_most<NK, kStep>(key, most);
        return false;
    };

    Sums<T, INTERP, CB> sums;
    auto add = [&](uint32_t k) {
        const uint32_t i = k & ((1u << kPosBits) - 1u);
        T go[GS];
        __builtin_memcpy(go, __builtin_assume_aligned(&s_go[i * GS], sizeof(T) * GS), sizeof(T) * GS);
        float w = 1.0f;
        if constexpr (INTERP == 0) {
            w = s_weight.get(i, (k >> kPosBits) & ((1u << DIM) - 1u));
        }
        // a contribution that is not there is zero times zero, which changes no sum that started at +0
        sums.add(go, w);
    };
    auto fold = [&]() {
#pragma unroll
        for (int g = 0; g < NK; g += kStep) {
            if (g < most) {
#pragma unroll
                for (int i = g; i < g + kStep; i++) {
                    add(key[i]);
                }
            }
        }
        const uint64_t rare = __builtin_amdgcn_ballot_w64(crowded);
        if (rare == 0) {
            return;
        }
        int lane = t & 63;
        asm volatile("" : "+v"(lane));  // what follows is rare: none of it is worked out ahead
        const uint32_t all = wave_sum(crowded ? len : 0u);
        const bool together = crowded && ((len > kSerialMost && len * kSideBySide > all) ||
                                          ((sorted & only) != kNoKey && __builtin_popcountll(rare) <= kFewCrowded));
        if (crowded && !together) {
            if (only != kNoKey) {
                for (uint32_t i = 0; i < len; i++) {
                    add(s_list[only + i] ^ corner);
                }
            } else if (sorted != kNoKey) {
                for (uint32_t i = 0; i < len; i++) {
                    add(s_sorted[sorted + i]);
                }
            } else {
                merge_alone([&](uint32_t, uint32_t k) { add(k); });
            }
        }
        // The wavefront together, an element after the other: 64 contributions at a time are computed side by side, and a
        // lane per channel adds them one by one.
        ByWave& own = s_rare.waves[wave];
        uint64_t big = __builtin_amdgcn_ballot_w64(together);
        while (big != 0) {
            const int owner = __builtin_ctzll(big);
            big &= big - 1u;
            float sum = 0.0f;  // of channel `lane`
#pragma unroll
            for (int j = 0; j < CB; j++) {
                const float s = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, sums.get(j)), owner));
                sum = (lane == j) ? s : sum;
            }
            auto add_batch = [&](uint32_t k, uint32_t batch) {  // k: lane's key, of the first where it has none
                const bool have = (uint32_t)lane < batch;
                const uint32_t i = k & ((1u << kPosBits) - 1u);
                float w = 1.0f;
                if constexpr (INTERP == 0) {
                    w = s_weight.get(i, (k >> kPosBits) & ((1u << DIM) - 1u));
                }
                bool some = false;
#pragma unroll
                for (int j = 0; j < CB; j++) {
                    const float v = have ? value_of<T, INTERP>(ElemIO<T>::load(&s_go[i * GS + j]), w) : 0.0f;
                    own.value[j][lane] = v;
                    some = some || v != 0.0f;
                }
                landed();
                // zeros change no sum: padding piles points up with weight 0 on the elements next to an edge
                if (__builtin_amdgcn_ballot_w64(some) != 0 && lane < CB) {
                    sum = add_in_order<T>(sum, own.value[lane], batch);
                }
                landed();
            };
            const uint32_t from = (uint32_t)__builtin_amdgcn_readlane((int)sorted, owner);
            const uint32_t run = (uint32_t)__builtin_amdgcn_readlane((int)only, owner);
            const uint32_t its_corner = (uint32_t)__builtin_amdgcn_readlane((int)corner, owner);
            const uint32_t its_len = (uint32_t)__builtin_amdgcn_readlane((int)len, owner);
            if ((from & run) != kNoKey) {
                auto key_of = [&](uint32_t done) {
                    const uint32_t i = done + (uint32_t)lane < its_len ? done + (uint32_t)lane : 0u;
                    return run != kNoKey ? s_list[run + i] ^ its_corner : (uint32_t)s_sorted[from + i];
                };
                uint32_t k = key_of(0u);
                for (uint32_t done = 0; done < its_len; done += 64u) {
                    const uint32_t next = key_of(done + 64u);
                    add_batch(k, its_len - done < 64u ? its_len - done : 64u);
                    k = next;
                }
            } else {
                merge_together(owner, lane, [&](uint32_t rank, uint32_t k) { own.order[rank] = (uint16_t)k; },
                               [&](uint32_t batch) {
                                   landed();
                                   add_batch(own.order[(uint32_t)lane < batch ? lane : 0], batch);
                               });
            }
#pragma unroll
            for (int j = 0; j < CB; j++) {
                const float s = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, sum), j));
                if (lane == owner) {
                    sums.set(j, s);
                }
            }
        }
    };

    // Runs of segments that fit LDS, in order; the channels in turn for each.  The sums so far are values of the element type
    // and wait in the gradient itself, where the lane that stored them reads them again.
    const bool inside = x0 + lx < p.W && y0 + ly < p.H && z0 + lz < p.D;
    const uint32_t e = (uint32_t)(((z0 + lz) * p.H + y0 + ly) * p.W + x0 + lx) * (uint32_t)sizeof(T);
    uint32_t from = 0;
    do {
        uint32_t to = segs;
        if (total - s_before[from] > (uint32_t)CAP) {
            uint32_t lo = from + 1u;  // the last that fits: a segment does
            while (to - lo > 1u) {
                const uint32_t mid = (lo + to) >> 1;
                if (s_before[mid] - s_before[from] <= (uint32_t)CAP) {
                    lo = mid;
                } else {
                    to = mid;
                }
            }
            to = lo;
        }
        for (int32_t c0 = c_begin; c0 < c_end; c0 += CB) {
            const int32_t nc = (c_end - c0 < CB) ? c_end - c0 : CB;
            char* out = reinterpret_cast<char*>(dx + ((int64_t)n * p.C + c0) * (int64_t)p.elements);
            auto at = [&](int j) { return reinterpret_cast<T*>(out + (int64_t)j * p.elements * (int64_t)sizeof(T) + e); };
            sums.clear();
            if (to > from) {
                if (c0 == c_begin) {
                    if (build(from, to, c0, nc)) {
                        leave();
                        return;
                    }
                } else {
                    T go[RPL][GS];
#pragma unroll
                    for (int k = 0; k < RPL; k++) {
                        if (lane_points(k)) {
                            load_go(c0, nc, k, go[k]);
                        }
                    }
#pragma unroll
                    for (int k = 0; k < RPL; k++) {
                        if (lane_points(k)) {
                            stage_go(k, go[k]);
                        }
                    }
                    __syncthreads();
                }
                if (from > 0u && inside) {
#pragma unroll
                    for (int j = 0; j < CB; j++) {
                        if (j < nc) {
                            sums.set(j, ElemIO<T>::load(at(j)));
                        }
                    }
                }
                fold();
            }
            if (inside) {
#pragma unroll
                for (int j = 0; j < CB; j++) {
                    if (j < nc) {
                        ElemIO<T>::store(at(j), sums.get(j));
                    }
                }
            }
            if (to < segs || c0 + CB < c_end) {
                __syncthreads();  // LDS is written again
            }
        }
        from = to;
    } while (from < segs);
}

inline uint32_t xcd_blocks(int64_t pieces) { return (uint32_t)((pieces + 7) / 8 * 8); }

template <typename T, int DIM, int INTERP, int GRID>
hipError_t launch_bin(const GradGatherArgs& a, const TilesPlan& pl, hipStream_t stream, const GridToo<DIM>& too, int64_t grid_blocks)
{
    static std::atomic<uint32_t> bin_allowed{0};
    const hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(gs_tiles_bin_kernel<T, DIM, INTERP, GRID>),
                                           (int)kTilesMost * (kBinThreads / 64) * 12, bin_allowed);
    if (e != hipSuccess) {
        return e;
    }
    const uint32_t bins = (uint32_t)a.N * (uint32_t)pl.p.blocks, blocks = xcd_blocks(bins);
    hipLaunchKernelGGL((gs_tiles_bin_kernel<T, DIM, INTERP, GRID>), dim3(blocks + (uint32_t)grid_blocks), dim3(kBinThreads),
                       (size_t)pl.bin_lds, stream, (const T*)a.grid, (uint32_t*)a.scratch, pl.p, bins, blocks, too);
    return hipGetLastError();
}

// The bin kernel, with the gradient of the whole batch's grid behind its workgroups where that is wanted (a.dgrid).
template <typename T, int DIM, int INTERP>
hipError_t run_bin(const GradGatherArgs& a, const TilesPlan& pl, hipStream_t stream)
{
    GridToo<DIM> too{};
    if (a.dgrid == nullptr) {
        return launch_bin<T, DIM, INTERP, 0>(a, pl, stream, too, 0);
    }
    too.gout = a.gout;
    too.x = a.x;
    too.dgrid = a.dgrid;
    if constexpr (DIM == 2) {
        const Grid2Launch g = grid2_launch(a);
        too.p = g.p;
        if constexpr (INTERP == 0) {
            if (g.tiled) {
                return launch_bin<T, DIM, INTERP, 2>(a, pl, stream, too, g.blocks);
            }
        }
        return launch_bin<T, DIM, INTERP, 1>(a, pl, stream, too, g.blocks);
    } else {
        too.p = grid3_params(a);
        const int64_t blocks = (too.p.total + kBinThreads - 1) / kBinThreads;
        return (INTERP == 0 && too.p.total < kGridGradFewPoints) ? launch_bin<T, DIM, INTERP, 2>(a, pl, stream, too, blocks)
                                                                 : launch_bin<T, DIM, INTERP, 1>(a, pl, stream, too, blocks);
    }
}

template <typename T, int DIM, int INTERP, int CB>
hipError_t launch_tiles(const GradGatherArgs& a, const TilesPlan& pl, hipStream_t stream)
{
    typedef GradTile<DIM> S;
    hipError_t e = hipSuccess;
    static std::atomic<uint32_t> gather_allowed{0};
    e = allow_dynamic_lds(reinterpret_cast<const void*>(gs_tiles_gather_kernel<T, DIM, INTERP, CB>),
                          (int)(kTileBlocksMost + 1) * 8, gather_allowed);
    if (e != hipSuccess) {
        return e;
    }
    e = run_bin<T, DIM, INTERP>(a, pl, stream);
    if (e != hipSuccess) {
        return e;
    }
    const uint32_t pieces = (uint32_t)a.N * pl.p.by_item.div;
    hipLaunchKernelGGL((gs_tiles_gather_kernel<T, DIM, INTERP, CB>), dim3(xcd_blocks(pieces)), dim3(S::kThreads),
                       (size_t)pl.segment_lds, stream, (const T*)a.gout, (const T*)a.grid, (T*)a.dx,
                       (const uint32_t*)a.scratch, (uint32_t*)a.scratch + pl.p.list, pl.p, pieces, pl.chans_per_block);
    e = hipGetLastError();
    return (e == hipSuccess && pl.p.list_most > 0) ? run_crowded_tiles(a, pl, stream) : e;
}

template <typename T, int DIM, int INTERP>
hipError_t run_channels(const GradGatherArgs& a, const TilesPlan& pl, hipStream_t stream)
{
    switch (pl.cb) {
        case 1: return launch_tiles<T, DIM, INTERP, 1>(a, pl, stream);
        case 2: return launch_tiles<T, DIM, INTERP, 2>(a, pl, stream);
        case 3: return launch_tiles<T, DIM, INTERP, 3>(a, pl, stream);
        case 4: return launch_tiles<T, DIM, INTERP, 4>(a, pl, stream);
        default: break;
    }
    if constexpr (sizeof(T) == 2 && DIM == 2) {
        return launch_tiles<T, DIM, INTERP, 8>(a, pl, stream);
    }
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t run_typed(const GradGatherArgs& a, const TilesPlan& pl, hipStream_t stream)
{
    switch (a.dim * 2 + a.interp) {
        case 2 * 2 + 0: return run_channels<T, 2, 0>(a, pl, stream);
        case 2 * 2 + 1: return run_channels<T, 2, 1>(a, pl, stream);
        case 3 * 2 + 0: return run_channels<T, 3, 0>(a, pl, stream);
        case 3 * 2 + 1: return run_channels<T, 3, 1>(a, pl, stream);
        default: return hipErrorInvalidValue;
    }
}

// Whether the bin kernel takes the gradient of the grid along: its workgroups have the bin's LDS too, which four and more a CU
// can have.
bool takes_grid(const GradGatherArgs& a, const TilesPlan& pl)
{
    if (a.dgrid == nullptr || a.x == nullptr || pl.group < a.N || pl.bin_lds > 40 * 1024) {
        return false;
    }
    const int64_t blocks = a.dim == 2 ? grid2_launch(a).blocks : (a.N * a.points + kBinThreads - 1) / kBinThreads;
    return fits_launch(blocks + a.N * (int64_t)pl.p.blocks + 16, kBinThreads);
}

}  // namespace

int64_t grad_tiles_words(const GradGatherArgs& a)
{
    const TilesPlan pl = tiles_plan(a);
    return pl.ok ? pl.words : 0;
}

hipError_t run_grad_tiles(const GradGatherArgs& a, hipStream_t stream, bool* dgrid_done)
{
    TilesPlan pl = tiles_plan(a);
    if (!pl.ok || a.dx == nullptr || a.gout == nullptr || a.grid == nullptr || a.scratch == nullptr) {
        return hipErrorInvalidValue;
    }
    // Items in one group: the bin kernel takes the gradient of the grid along.
    const bool take_grid = takes_grid(a, pl);
    // the items are independent: a group of them after the other, each in all of the scratch
    const int64_t esz = elem_size(a.elem);
    for (int64_t first = 0; first < a.N; first += pl.group) {
        GradGatherArgs g = a;
        g.dgrid = take_grid ? a.dgrid : nullptr;
        g.N = (a.N - first < pl.group) ? a.N - first : pl.group;
        g.gout = (const char*)a.gout + first * a.C * a.points * esz;
        g.grid = (const char*)a.grid + first * a.points * a.dim * esz;
        g.dx = (char*)a.dx + first * a.C * (a.D * a.H * a.W) * esz;
        pl.p.N = (int32_t)g.N;
        pl.p.first_item = (int32_t)first;
        hipError_t e = hipErrorInvalidValue;
        switch (a.elem) {
            case Elem::F32: e = run_typed<float>(g, pl, stream); break;
            case Elem::F16: e = run_typed<_Float16>(g, pl, stream); break;
            case Elem::BF16: e = run_typed<__bf16>(g, pl, stream); break;
        }
        if (e != hipSuccess) {
            return e;
        }
    }
    *dgrid_done = *dgrid_done || take_grid;
    return hipSuccess;
}

}  // namespace opscv
