// Input gradient by tiles (gs_grad_tiles.hip): the tiles that many points fall on.  The same sums in the same order.
//
// A grid over a part of the plane or volume puts all of an item's points on few tiles.  A workgroup per tile would take them
// round after round, 15 us each and up to 350 where every element has hundreds of contributions, while the rest of the chip has
// nothing to do.  gs_tiles_gather_kernel leaves tiles beyond TilesParams::crowded points on a list, and here a workgroup takes
// a part of such a tile (8 x 4 elements of a plane, 4 x 4 x 4 of a volume) and some channels:
//
//   select  the tile's points, in order; a record says in which part of the tile its corners lie, so that most points cost a
//           record of two bytes and no more
//   rank    a wavefront takes a chunk of 256 grid points at a time: the place of every point among those of its cell in the
//           chunk, and how many each cell has
//   place   sums over the counts give where an element's contributions from a chunk begin, and within it those of every tap:
//           the sequence is (chunk, tap, point)
//   add     a lane per element and channel, its contributions one by one in that order
//
// Bound by the chain of steps of a round, 10 to 15 us for 512 points (2048 of nearest samples): fp32 1x3x480x640 from as many
// points on an eighth of either axis 147 us, without the adds 141, without placing 138, without ranks 128.  The contributions
// lie in LDS as values in order: as places of weights and gradients, three loads each, a spot of 55000 points took 5.3 ms, 1.4
// so.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "gs_grad_gather.hpp"
#include "gs_grad_points.hpp"
#include "gs_grad_tiles_kernel.hpp"
#include "gs_grad_tiles_plan.hpp"
#include "kernels.hpp"

namespace opscv {

namespace {

constexpr int kCrowdThreads = 256;
constexpr int kCellBits = 7;
constexpr int kAhead = 8;          // contributions that a lane loads ahead
constexpr int kLook = 8;           // records that a lane looks at together

// Channels of a workgroup: as many as the contributions of a round leave room for (35 KiB; three workgroups per CU).
template <typename T, int DIM>
constexpr int crowd_channels()
{
    return (DIM == 3 && sizeof(T) == 4) ? 2 : 4;
}

// the weight of corner `tap` of a point's cell: weight_of(), which is given the corner
template <typename T, int DIM, int INTERP>
__device__ __forceinline__ float corner_weight(const Coords<T, DIM>& c, int tap)
{
    if constexpr (INTERP == 1) {
        return 1.0f;
    }
    float w = 0.0f;
#pragma unroll
    for (int k = 0; k < DIM; k++) {
        const float f = ElemIO<T>::load(&c.v[k]), low = __builtin_floorf(f), d = ((tap >> k) & 1) ? f - low : (low + 1.0f) - f;
        w = (k == 0) ? d : w * d;
    }
    return rt<T>(as_fp32_value(w));
}

template <typename T, int DIM, int INTERP>
__global__ __launch_bounds__(kCrowdThreads) void gs_tiles_crowded_kernel(const T* __restrict__ gout, const T* __restrict__ grid,
                                                                         T* __restrict__ dx, const uint32_t* __restrict__ ws,
                                                                         TilesParams p, int32_t cgroups)
{
    typedef GradTile<DIM> S;
    // points in LDS: two chunks at least, so that one of them is whole; more of nearest samples, whose points are one contribution
    constexpr int kCrowdPoints = (INTERP == 1) ? 2048 : 512;
    constexpr int TH = kCrowdThreads, kWaves = TH / 64, kOwn = kCrowdPoints / TH, kStrips = kCrowdPoints / 64;
    constexpr int EX = S::kPartX, EY = S::kPartY, EZ = S::kPartZ, kElements = EX * EY * EZ, kChannels = crowd_channels<T, DIM>();
    constexpr int kPartsX = S::kX / EX, kPartsY = S::kY / EY, kPartsZ = S::kZ / EZ, kParts = kPartsX * kPartsY * kPartsZ;
    constexpr int PADC = (INTERP == 0) ? 1 : 0;
    constexpr int CX = EX + PADC, CY = EY + PADC, CZ = (DIM == 3) ? EZ + PADC : 1, CELLS = CX * CY * CZ;
    constexpr int K = (INTERP == 0) ? (1 << DIM) : 1;  // taps of a point, cells of an element
    constexpr int kChunks = 4 * TH / kElements;         // of a round at most
    constexpr int kValues = K * kCrowdPoints + 2 * kAhead;  // contributions of a channel; lanes read past their own
    constexpr int kCounts = kChunks * CELLS;
    static_assert(kParts <= (1 << kRecordPartBits) && kBinPoints == (1 << kRecordBits), "fields of a record");
    static_assert(CELLS <= (1 << kCellBits) && kCrowdPoints >= 2 * 256, "fields of a point");
    static_assert(kStrips <= kLook * kWaves && kStrips <= 64, "counts of the strips");
    __shared__ uint32_t s_point[kCrowdPoints];  // block << 10 | number within it
    __shared__ uint8_t s_cell[kCrowdPoints];
    __shared__ uint16_t s_rank[kCrowdPoints];   // among the chunk's points of its cell
    __shared__ uint8_t s_chunk[kCrowdPoints];
    __shared__ uint16_t s_begin[kCrowdPoints + 1];  // of every chunk
    __shared__ uint32_t s_count[kCounts];       // [chunk][cell]
    __shared__ __align__(16) uint32_t s_first[kElements * kChunks];  // [element][chunk]: the first contribution
    __shared__ T s_value[kChannels * kValues];  // of every channel, an element after the other, in order
    __shared__ uint32_t s_found[2][kLook * kWaves];
    __shared__ uint32_t s_scan[kWaves], s_total;
    extern __shared__ uint32_t s_seg[];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    uint32_t* s_before = s_seg;
    uint32_t* s_where = s_seg + p.blocks + 1;
    const uint32_t listed = ws[p.list] < p.list_most ? ws[p.list] : p.list_most;
    const int64_t parts = (int64_t)listed * kParts * cgroups;
    // the lane's element of the part, and its channel (lanes beyond the channels add nothing)
    const int e = t % kElements, own_channel = t / kElements;
    // the cell of which element x, y, z of the part is corner `tap`
    auto cell_of_tap = [](int x, int y, int z, int tap) {
        return INTERP == 1 ? (z * CY + y) * CX + x
                           : ((DIM == 3 ? z + 1 - (tap >> 2) : 0) * CY + y + 1 - ((tap >> 1) & 1)) * CX + x + 1 - (tap & 1);
    };

    for (int64_t part = blockIdx.x; part < parts; part += gridDim.x) {
        const int32_t c0 = (int32_t)(part % cgroups) * kChannels;
        const int32_t nc = (p.C - c0 < kChannels) ? p.C - c0 : kChannels;
        const uint32_t sub = (uint32_t)(part / cgroups % kParts);
        const uint32_t entry = ws[p.list + 1u + (uint32_t)(part / cgroups / kParts)];
        const uint32_t n = entry >> kTileBits, tile = entry & ((1u << kTileBits) - 1u);
        const int32_t tile_yz = (int32_t)fast_div(tile, p.by_tiles_x), tile_x = (int32_t)tile - tile_yz * p.tiles_x;
        const int32_t tile_z = (DIM == 3) ? (int32_t)fast_div((uint32_t)tile_yz, p.by_tiles_y) : 0;
        const int32_t tile_y = tile_yz - tile_z * p.tiles_y;
        const uint32_t sx = sub % kPartsX, sy = sub / kPartsX % kPartsY, sz = sub / (kPartsX * kPartsY);
        const int32_t x0 = tile_x * S::kX + (int32_t)sx * EX, y0 = tile_y * S::kY + (int32_t)sy * EY;
        const int32_t z0 = tile_z * S::kZ + (int32_t)sz * EZ;
        if (x0 >= p.W || y0 >= p.H || z0 >= p.D) {
            continue;
        }
        const int32_t phase = (DIM == 3 && p.items_per_core > 1) ? phase_of(n, p) : 0;
        const uint32_t* item = ws + (size_t)n * p.lay.item_words;
        const uint16_t* records = reinterpret_cast<const uint16_t*>(item + p.lay.records);
        const T* go_n = gout + ((int64_t)n * p.C + c0) * (int64_t)p.points;
        const T* grid_n = grid + (int64_t)n * p.points * DIM;
        uint32_t segs, total;
        __syncthreads();  // the part before is done with LDS
        tile_segments<TH>(item, p, tile, s_before, s_where, s_scan, &segs, &total);
        __syncthreads();

        uint32_t have = 0;  // points in LDS
        float sum = 0.0f;
        // A round: whole chunks of the points in LDS, and not the last one, which may go on behind them, unless this is the end.
        auto add_points = [&](bool end) {
            uint32_t point[kOwn], begins[kOwn], cell[kOwn];
            Coords<T, DIM> coords[kOwn];
            T raw[kOwn][DIM], go[kOwn][kChannels];
            for (int i = t; i < kCounts; i += TH) {
                s_count[i] = 0u;
            }
            __syncthreads();
#pragma unroll
            for (int u = 0; u < kOwn; u++) {
                const uint32_t i = (uint32_t)(u * TH + t);
                point[u] = s_point[i < have ? i : 0u];
                const int32_t pt = (int32_t)point[u] - phase;
                __builtin_memcpy(raw[u], grid_n + (int64_t)pt * DIM, sizeof(raw[u]));
#pragma unroll
                for (int j = 0; j < kChannels; j++) {
                    go[u][j] = go_n[(int64_t)(j < nc ? j : 0) * p.points + pt];
                }
                const uint32_t left = s_point[(i < have && i > 0u) ? i - 1u : 0u];
                const bool is = i < have && (i == 0u || (left >> 8) != (point[u] >> 8));
                const uint64_t mask = __builtin_amdgcn_ballot_w64(is);
                begins[u] = bits_below(mask) + (is ? 1u : 0u);  // of the strip's, up to here
                if (lane == 0) {
                    s_found[0][u * kWaves + wave] = (uint32_t)__builtin_popcountll(mask);
                }
            }
            __syncthreads();
            const uint32_t of_strip = (lane < kStrips) ? s_found[0][lane < kStrips ? lane : 0] : 0u;
            const uint32_t strips = wave_scan(of_strip), chunks = (uint32_t)__builtin_amdgcn_readlane((int)strips, kStrips - 1);
#pragma unroll
            for (int u = 0; u < kOwn; u++) {
                const uint32_t i = (uint32_t)(u * TH + t), left = s_point[(i < have && i > 0u) ? i - 1u : 0u];
                const uint32_t chunk = begins[u] + (uint32_t)__builtin_amdgcn_readlane((int)(strips - of_strip), u * kWaves + wave) - 1u;
                if (i < have) {
                    coords[u] = coords_of<T, DIM, INTERP>(raw[u], p);
                    int32_t x, y, z;
                    low_corner<T, DIM, INTERP>(coords[u], p, &x, &y, &z);
                    x += PADC - x0;
                    y += PADC - y0;
                    z += (DIM == 3) ? PADC - z0 : 0;
                    cell[u] = (uint32_t)((z * CY + y) * CX + x);
                    cell[u] = cell[u] < (uint32_t)CELLS ? cell[u] : 0u;  // always: its record says so
                    s_cell[i] = (uint8_t)cell[u];
                    s_chunk[i] = (uint8_t)chunk;
                    if (i == 0u || (left >> 8) != (point[u] >> 8)) {
                        s_begin[chunk] = (uint16_t)i;
                    }
                }
            }
            if (t == 0) {
                s_begin[chunks] = (uint16_t)have;
            }
            __syncthreads();
            uint32_t whole = end ? chunks : chunks - 1u;
            whole = whole < (uint32_t)kChunks ? whole : (uint32_t)kChunks;
            const uint32_t number = s_begin[whole];
            for (uint32_t c = (uint32_t)wave; c < whole; c += kWaves) {
                uint32_t* counts = s_count + c * CELLS;
                const uint32_t to = s_begin[c + 1u];
                for (uint32_t i0 = s_begin[c]; i0 < to; i0 += 64u) {
                    const uint32_t i = i0 + (uint32_t)lane;
                    const uint32_t cell = s_cell[i < to ? i : i0];
                    uint64_t same = __builtin_amdgcn_ballot_w64(i < to);
#pragma unroll
                    for (int b = 0; b < kCellBits; b++) {
                        const bool one = (cell >> b) & 1u;
                        const uint64_t ones = __builtin_amdgcn_ballot_w64(one);
                        same &= one ? ones : ~ones;
                    }
                    const uint32_t before = counts[cell], below = bits_below(same);
                    landed();
                    if (i < to) {
                        s_rank[i] = (uint16_t)(before + below);
                        if (below == 0u) {
                            counts[cell] = before + (uint32_t)__builtin_popcountll(same);
                        }
                    }
                    landed();
                }
            }
            __syncthreads();
            // four of an element's chunks a lane
            {
                const int el = t * 4 / kChunks, x = el % EX, y = el / EX % EY, z = el / (EX * EY);
                uint32_t len[4] = {0u, 0u, 0u, 0u};
#pragma unroll
                for (int c = 0; c < 4; c++) {
#pragma unroll
                    for (int k = 0; k < K; k++) {
                        len[c] += s_count[(t * 4 % kChunks + c) * CELLS + cell_of_tap(x, y, z, k)];
                    }
                }
                const uint32_t own = len[0] + len[1] + len[2] + len[3], incl = wave_scan(own);
                if (lane == 63) {
                    s_scan[wave] = incl;
                }
                __syncthreads();
                uint32_t all;
                const uint32_t at = sums_before<kWaves>(s_scan, wave, lane, &all) + incl - own;
                reinterpret_cast<uint4*>(s_first)[t] = make_uint4(at, at + len[0], at + len[0] + len[1], at + len[0] + len[1] + len[2]);
                if (t == 0) {
                    s_total = all;
                }
            }
            __syncthreads();
#pragma unroll
            for (int u = 0; u < kOwn; u++) {
                const uint32_t i = (uint32_t)(u * TH + t);
                if (i < number) {
                    const int cx = (int)cell[u] % CX, cy = (int)cell[u] / CX % CY, cz = (int)cell[u] / (CX * CY);
                    const uint32_t chunk = s_chunk[i], rank = s_rank[i];
                    const uint32_t* counts = s_count + chunk * CELLS;
#pragma unroll
                    for (int k = 0; k < K; k++) {
                        // the element that is corner k
                        const int x = cx - PADC + (k & 1), y = cy - PADC + ((k >> 1) & 1);
                        const int z = (DIM == 3) ? cz - PADC + (k >> 2) : 0;
                        if (x >= 0 && x < EX && y >= 0 && y < EY && z >= 0 && z < EZ) {
                            uint32_t at = s_first[((z * EY + y) * EX + x) * kChunks + chunk] + rank;
#pragma unroll
                            for (int o = 0; o < k; o++) {
                                at += counts[cell_of_tap(x, y, z, o)];
                            }
                            const float w = corner_weight<T, DIM, INTERP>(coords[u], k);
#pragma unroll
                            for (int j = 0; j < kChannels; j++) {
                                if (j < nc) {
                                    ElemIO<T>::store(&s_value[j * kValues + at], value_of<T, INTERP>(ElemIO<T>::load(&go[u][j]), w));
                                }
                            }
                        }
                    }
                }
            }
            __syncthreads();
            if (own_channel < nc) {
                uint32_t i = s_first[e * kChunks];
                const uint32_t to = (e + 1 < kElements) ? s_first[(e + 1 < kElements ? e + 1 : 0) * kChunks] : s_total;
                const T* values = s_value + own_channel * kValues;
                T v[kAhead];
                __builtin_memcpy(v, values + i, sizeof(v));
                while (i + kAhead <= to) {
                    T next[kAhead];
                    i += kAhead;
                    __builtin_memcpy(next, values + i, sizeof(next));
#pragma unroll
                    for (int k = 0; k < kAhead; k++) {
                        sum = rt<T>(sum + ElemIO<T>::load(&v[k]));
                        v[k] = next[k];
                    }
                }
#pragma unroll
                for (int k = 0; k < kAhead; k++) {
                    sum = (i + k < to) ? rt<T>(sum + ElemIO<T>::load(&v[k])) : sum;
                }
            }
            __syncthreads();
            // what is left to the front
            have -= number;
#pragma unroll
            for (int u = 0; u < kOwn; u++) {
                const uint32_t i = (uint32_t)(u * TH + t);
                point[u] = s_point[i < have ? number + i : 0u];
            }
            __syncthreads();
#pragma unroll
            for (int u = 0; u < kOwn; u++) {
                const uint32_t i = (uint32_t)(u * TH + t);
                if (i < have) {
                    s_point[i] = point[u];
                }
            }
            __syncthreads();
        };

        uint32_t steps = 1;
        while (steps < segs) {
            steps <<= 1;
        }
        uint32_t q[kLook], record[kLook];  // of the step to come: the first point of the block, the record
        auto look = [&](uint32_t i0) {
#pragma unroll
            for (int k = 0; k < kLook; k++) {
                uint32_t i = i0 + (uint32_t)(k * TH + t);
                i = i < total ? i : total - 1u;
                uint32_t seg = 0;  // the last segment that does not start behind point i
                for (uint32_t d = steps >> 1; d > 0u; d >>= 1) {
                    const uint32_t mid = seg + d < segs ? seg + d : segs;
                    seg = s_before[mid] <= i ? mid : seg;
                }
                const uint32_t where = s_where[seg], block = where >> 14;
                q[k] = block * kBinPoints;
                record[k] = records[(size_t)block * (p.lay.block_words * 2u) + (where & 0x3FFFu) + (i - s_before[seg])];
            }
        };
        look(0u);
        uint32_t turn = 0;
        for (uint32_t i0 = 0; i0 < total; i0 += kLook * TH, turn ^= 1u) {
            uint32_t own[kLook], at[kLook];
            bool takes[kLook];
#pragma unroll
            for (int k = 0; k < kLook; k++) {
                const uint32_t code = record[k] >> kRecordBits, low = code & ((1u << kRecordPartBits) - 1u);
                auto reaches = [&](uint32_t first, uint32_t mine, int axis) {
                    return first == mine || (((code >> (kRecordPartBits + axis)) & 1u) && first + 1u == mine);
                };
                takes[k] = i0 + (uint32_t)(k * TH + t) < total && reaches(low % kPartsX, sx, 0) &&
                           reaches(low / kPartsX % kPartsY, sy, 1) && (kPartsZ == 1 || reaches(low / (kPartsX * kPartsY), sz, 2));
                own[k] = q[k] + (record[k] & (kBinPoints - 1u));
                const uint64_t mask = __builtin_amdgcn_ballot_w64(takes[k]);
                at[k] = bits_below(mask);
                if (lane == 0) {
                    s_found[turn][k * kWaves + wave] = (uint32_t)__builtin_popcountll(mask);
                }
            }
            __syncthreads();
            const uint32_t found = (lane < kLook * kWaves) ? s_found[turn][lane < kLook * kWaves ? lane : 0] : 0u;
            const uint32_t before = wave_scan(found) - found;
#pragma unroll
            for (int k = 0; k < kLook; k++) {
                at[k] += (uint32_t)__builtin_amdgcn_readlane((int)before, k * kWaves + wave);
            }
            const uint32_t all = (uint32_t)__builtin_amdgcn_readlane((int)(before + found), kLook * kWaves - 1);
            look(i0 + kLook * TH);
            uint32_t done = 0;
            while (done < all) {
                const uint32_t room = kCrowdPoints - have, take = all - done < room ? all - done : room;
#pragma unroll
                for (int k = 0; k < kLook; k++) {
                    if (takes[k] && at[k] >= done && at[k] - done < take) {
                        s_point[have + at[k] - done] = own[k];
                    }
                }
                have += take;
                done += take;
                if (have == (uint32_t)kCrowdPoints) {
                    add_points(false);
                }
            }
        }
        while (have > 0u) {
            add_points(true);
        }
        const int ex = e % EX, ey = e / EX % EY, ez = e / (EX * EY);
        const int32_t x = x0 + ex, y = y0 + ey, z = z0 + ez;
        if (own_channel < nc && x < p.W && y < p.H && z < p.D) {
            T* out = dx + ((int64_t)n * p.C + c0 + own_channel) * (int64_t)p.elements;
            ElemIO<T>::store(out + ((int64_t)z * p.H + y) * p.W + x, sum);
        }
    }
}

template <typename T, int DIM, int INTERP>
hipError_t launch(const GradGatherArgs& a, const TilesPlan& pl, hipStream_t stream)
{
    typedef GradTile<DIM> S;
    constexpr int kElements = S::kPartX * S::kPartY * S::kPartZ, kChannels = crowd_channels<T, DIM>();
    static std::atomic<uint32_t> allowed{0};
    hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(gs_tiles_crowded_kernel<T, DIM, INTERP>),
                                     (int)(kTileBlocksMost + 1) * 8, allowed);
    if (e != hipSuccess) {
        return e;
    }
    const int32_t cgroups = (int32_t)((a.C + kChannels - 1) / kChannels);
    const int64_t most = (int64_t)pl.p.list_most * (S::kThreads / kElements) * cgroups;
    hipLaunchKernelGGL((gs_tiles_crowded_kernel<T, DIM, INTERP>), dim3((unsigned)(most < kCrowdedGroups ? most : kCrowdedGroups)),
                       dim3(kCrowdThreads), (size_t)pl.segment_lds, stream, (const T*)a.gout, (const T*)a.grid, (T*)a.dx,
                       (const uint32_t*)a.scratch, pl.p, cgroups);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_typed(const GradGatherArgs& a, const TilesPlan& pl, hipStream_t stream)
{
    switch (a.dim * 2 + a.interp) {
        case 2 * 2 + 0: return launch<T, 2, 0>(a, pl, stream);
        case 2 * 2 + 1: return launch<T, 2, 1>(a, pl, stream);
        case 3 * 2 + 0: return launch<T, 3, 0>(a, pl, stream);
        case 3 * 2 + 1: return launch<T, 3, 1>(a, pl, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

hipError_t run_crowded_tiles(const GradGatherArgs& a, const TilesPlan& pl, hipStream_t stream)
{
    switch (a.elem) {
        case Elem::F32: return launch_typed<float>(a, pl, stream);
        case Elem::F16: return launch_typed<_Float16>(a, pl, stream);
        case Elem::BF16: return launch_typed<__bf16>(a, pl, stream);
    }
    return hipErrorInvalidValue;
}

}  // namespace opscv
