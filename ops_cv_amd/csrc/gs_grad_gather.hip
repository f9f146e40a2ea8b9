// Backward of the grid samplers for gfx950: gradient of the input as a gather over lists of contributions, for planes
// and volumes of any size, every interpolation mode and any number of grid points.
//
// The sum that reaches an element of the gradient is a fixed sequence (gs2d_grad.hip, gs3d_grad.hip): its contributions
// ordered by (chunk of 256 grid points, tap, point), every add rounded to the element type.  The kernels there walk the
// chunks in order and elect, round after round, who may add to an element; every band of a plane looks at every chunk,
// so their time grows with points times plane elements.  Here the order is restored per element by sorting:
//
//   clear   the counts of every cell
//   count   one lane per grid point: an atomic count per cell gives the point its rank in the cell (which rank depends
//           on timing, which points a cell holds does not); the source coordinates go to scratch
//   place   one lane per eight cells: every cell gets a run of the item's list (a prefix sum per workgroup, one atomic
//           add per workgroup for its base: the order of the runs does not matter)
//   fill    one lane per grid point: the point's entry goes to its run
//   gather  one lane per element: the element collects the entries of the cells it is a corner of -- cell (y - ys,
//           x - xs) holds the points it is corner (ys, xs) of -- keyed (chunk, tap, point), sorts up to 16 or 32 of them in
//           registers and folds gradOutput times weight in that order with the reference's roundings, every channel
//           from the same list.  Elements with more contributions (border padding piles points up on the edges) go to a
//           list of their own; meanwhile spare workgroups sort the runs of more than 64 entries.
//   crowded one wavefront per listed element: puts up to 128 contributions in order by counting the lesser keys of each, more
//           by merging the element's runs, 64 entries at a time; the lanes compute the 64 contributions of a channel at
//           once and one lane adds them up in the reference's order.
//           A chain of waits, so everything that does not depend on the sums is on its way before them: the runs' next
//           entries, the next channels' gradOutput, the operands of the additions; the places of two runs' entries in
//           each other are found together, in as many steps as the longer one takes.  Both gradients, every step waited for in
//           turn / so, border padding: fp32 4x2x600x736 721 / 440 us, 3x1x520x609 -> 605x708 1031 / 674, 4x2x301x505 378 / 268,
//           3x3x210x328 182 / 132, fp16 2x4x360x552 95 / 82; nearest fp32 3x2x304x576 222 / 144.
//           Dense grids have many elements of a few contributions more than a list, where the steps of full runs were most
//           of the time.  This kernel, every step in turn / always steps for 64 entries and 64 additions / so: fp16 5x3x41x32x44
//           -> 57x45x62 reflection 134 / 225 / 74, 22x2x10x85x61 -> 14x125x89 1254 / 1801 / 609, fp32 12x3x32x58x57 ->
//           39x71x69 border 251 / 317 / 107; bicubic (one run) 1x3x231x430 -> 323x602 138 / 217 / 116.
//
// Input gradient of fp32 8x3x479x637 from as many grid points (rotations of up to 30 degrees): 2568 us with elections;
// here clear 6, count 43, place 14, fill 13, gather 107, crowded 5 us.  Count is bound by the rate of atomics (55 G/s;
// four points per lane in flight or one, no difference), gather by the loads it issues per element (about fifty per
// wavefront: two starts, two counts, two entries per cell, then coordinates and gradOutput per contribution) beside the
// sorting network's instructions: twice the wavefronts in flight (lists of 16 instead of 32) leave its time as it is.
//
// A cell is an element of the lattice of low corners for linear interpolation (one entry per point, 2^DIM runs per
// element), and the element itself for nearest (one entry per point) and bicubic (sixteen entries per point: padding
// is applied tap by tap, so a tap's element does not follow from the point's cell).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "gs_grad_gather.hpp"
#include "gs_grad_points.hpp"
#include "gs_grad_sort_list.hpp"
#include "kernels.hpp"

namespace opscv {

namespace {

constexpr int kThreads = kGatherThreads;
constexpr int kPlaceCells = 8;       // cells per lane of the place kernel
constexpr int kPlaceThreads = 256;
constexpr int kFoldPitch = 68;       // of a channel's contributions in LDS: on the 16-byte grid, channels at different banks
constexpr int kFoldChans = 16;       // channels whose contributions a crowded element's wavefront computes together
constexpr uint32_t kCountedMost = 128;  // contributions of several runs that are put in order by counting, longer ones by merging
constexpr uint32_t kNoRank = 0xFFFFFFFFu;

// Grid points per lane of the count and fill kernels: the atomics and the scattered stores of several are on their way
// together.
template <int DIM, int INTERP>
constexpr int points_per_lane()
{
    return (INTERP == 2) ? 1 : 4;
}

// What depends on the mode: runs an element merges, entries a point makes, how an entry and a run make a sorting key
// (ascending keys are the reference's order) and back.  An entry is q = point + phase of the item's first chunk, with
// the tap between chunk and point for bicubic.
template <int DIM, int INTERP>
struct Mode {
    static constexpr int kRuns = (INTERP == 0) ? (1 << DIM) : 1;
    static constexpr int kEntries = (INTERP == 2) ? 16 : 1;
    static constexpr int kTapBits = (INTERP == 0) ? DIM : ((INTERP == 2) ? 4 : 0);
    static __device__ __forceinline__ uint32_t key(uint32_t entry, uint32_t run)
    {
        return (INTERP == 0) ? ((entry >> 8) << (8 + DIM)) | (run << 8) | (entry & 255u) : entry;
    }
    static __device__ __forceinline__ uint32_t entry(uint32_t q, uint32_t tap)
    {
        return (INTERP == 2) ? ((q >> 8) << 12) | (tap << 8) | (q & 255u) : q;
    }
    static __device__ __forceinline__ uint32_t tap_of(uint32_t key)
    {
        return (kTapBits > 0) ? (key >> 8) & ((1u << kTapBits) - 1u) : 0u;
    }
    static __device__ __forceinline__ uint32_t q_of(uint32_t key)
    {
        return (kTapBits > 0) ? ((key >> (8 + kTapBits)) << 8) | (key & 255u) : key;
    }
};

// Calls f(entry number, tap, cell) for every entry that the point makes.
template <typename T, int DIM, int INTERP, typename F>
__device__ __forceinline__ void for_entries(const Coords<T, DIM>& c, const GatherParams& p, F&& f)
{
    const float fx = ElemIO<T>::load(&c.v[0]), fy = ElemIO<T>::load(&c.v[1]);
    if constexpr (INTERP == 2) {
        const float xf = __builtin_floorf(fx), yf = __builtin_floorf(fy);
#pragma unroll
        for (int i = 0; i < 4; i++) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int32_t off = bicubic_bounded_offset(xf - 1.0f + (float)i, yf - 1.0f + (float)j, p.W, p.H, p.pad,
                                                           p.align);
                f(i * 4 + j, off);
            }
        }
    } else if constexpr (INTERP == 1) {
        const int32_t x = float_to_i32(__builtin_rintf(fx)), y = float_to_i32(__builtin_rintf(fy));
        int32_t z = 0;
        if constexpr (DIM == 3) {
            z = float_to_i32(__builtin_rintf(ElemIO<T>::load(&c.v[2])));
        }
        const bool in = (uint32_t)x < (uint32_t)p.W && (uint32_t)y < (uint32_t)p.H && (uint32_t)z < (uint32_t)p.D;
        f(0, in ? (z * p.H + y) * p.W + x : -1);
    } else {
        const int32_t x = float_to_i32(__builtin_floorf(fx)), y = float_to_i32(__builtin_floorf(fy));
        int32_t z = -1;
        if constexpr (DIM == 3) {
            z = float_to_i32(__builtin_floorf(ElemIO<T>::load(&c.v[2])));
        }
        // a point none of whose corners is inside has no cell
        const bool in = x >= -1 && x < p.W && y >= -1 && y < p.H && z >= -1 && z < p.D;
        f(0, in ? ((z + 1) * (p.H + 1) + (y + 1)) * (p.W + 1) + (x + 1) : -1);
    }
}

__global__ __launch_bounds__(kThreads) void gs_gather_clear_kernel(uint32_t* __restrict__ ws, uint32_t words,
                                                                    uint32_t item_words)
{
    uint32_t* wsn = ws + (size_t)blockIdx.y * item_words;
    const uint32_t i = (blockIdx.x * kThreads + threadIdx.x) * 4u;
    if (i < words) {  // whole units: the words behind the counts are written later anyway
        *reinterpret_cast<uint4*>(wsn + i) = make_uint4(0u, 0u, 0u, 0u);
    }
}

template <typename T, int DIM, int INTERP>
__global__ __launch_bounds__(kThreads) void gs_gather_count_kernel(const T* __restrict__ grid, uint32_t* __restrict__ ws,
                                                                    GatherParams p, uint32_t pieces, uint32_t per_item)
{
    constexpr int PPL = points_per_lane<DIM, INTERP>();
    constexpr int NE = Mode<DIM, INTERP>::kEntries;
    uint32_t n, local;
    if (!piece_of_block(blockIdx.x, pieces, per_item, &n, &local)) {
        return;
    }
    const int32_t first = (int32_t)(local * kThreads * PPL + threadIdx.x);
    uint32_t* wsn = ws + (size_t)n * p.lay.item_words;
    Coords<T, DIM> c[PPL];
#pragma unroll
    for (int u = 0; u < PPL; u++) {
        const int32_t pt = first + u * kThreads;
        c[u] = coords_of<T, DIM, INTERP>(grid + ((int64_t)n * p.points + (pt < p.points ? pt : 0)) * DIM, p);
    }
    uint32_t rank[PPL][NE];
#pragma unroll
    for (int u = 0; u < PPL; u++) {
        const bool have = first + u * kThreads < p.points;
        for_entries<T, DIM, INTERP>(c[u], p, [&](int i, int32_t cell) {
            rank[u][i] = (have && cell >= 0) ? atomicAdd(&wsn[p.lay.counts + cell], 1u) : kNoRank;
        });
    }
#pragma unroll
    for (int u = 0; u < PPL; u++) {
        const int32_t pt = first + u * kThreads;
        if (pt < p.points) {
            reinterpret_cast<Coords<T, DIM>*>(wsn + p.lay.coords)[pt] = c[u];
#pragma unroll
            for (int i = 0; i < NE; i++) {
                wsn[p.lay.ranks + (size_t)i * p.points + pt] = rank[u][i];
            }
        }
    }
}

__global__ __launch_bounds__(kPlaceThreads) void gs_gather_place_kernel(uint32_t* __restrict__ ws, GatherParams p)
{
    __shared__ uint32_t s_sum[kPlaceThreads / 64];
    __shared__ uint32_t s_base;
    uint32_t* wsn = ws + (size_t)blockIdx.y * p.lay.item_words;
    const int t = threadIdx.x;
    const int32_t first = (int32_t)((blockIdx.x * kPlaceThreads + t) * kPlaceCells);
    uint32_t cnt[kPlaceCells], sum = 0;
#pragma unroll
    for (int i = 0; i < kPlaceCells; i++) {
        cnt[i] = (first + i < p.cells) ? wsn[p.lay.counts + first + i] : 0u;
        sum += cnt[i];
    }
    uint32_t incl = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t up = __shfl_up(incl, d);
        incl += ((t & 63) >= d) ? up : 0u;
    }
    if ((t & 63) == 63) {
        s_sum[t >> 6] = incl;
    }
    __syncthreads();
    if (t == 0) {
        uint32_t total = 0;
        for (int w = 0; w < kPlaceThreads / 64; w++) {
            const uint32_t s = s_sum[w];
            s_sum[w] = total;
            total += s;
        }
        s_base = atomicAdd(&wsn[0], total);
    }
    __syncthreads();
    uint32_t at = s_base + s_sum[t >> 6] + incl - sum;
#pragma unroll
    for (int i = 0; i < kPlaceCells; i++) {
        if (first + i < p.cells) {
            wsn[p.lay.starts + first + i] = at;
            at += cnt[i];
            if (cnt[i] > kSortedRun) {
                wsn[p.lay.runs + atomicAdd(&wsn[1], 1u)] = (uint32_t)(first + i);
            }
        }
    }
}

template <typename T, int DIM, int INTERP>
__global__ __launch_bounds__(kThreads) void gs_gather_fill_kernel(uint32_t* __restrict__ ws, GatherParams p,
                                                                   uint32_t pieces, uint32_t per_item)
{
    constexpr int PPL = points_per_lane<DIM, INTERP>();
    constexpr int NE = Mode<DIM, INTERP>::kEntries;
    uint32_t n, local;
    if (!piece_of_block(blockIdx.x, pieces, per_item, &n, &local)) {
        return;
    }
    const int32_t first = (int32_t)(local * kThreads * PPL + threadIdx.x);
    uint32_t* wsn = ws + (size_t)n * p.lay.item_words;
    Coords<T, DIM> c[PPL];
    uint32_t rank[PPL][NE];
#pragma unroll
    for (int u = 0; u < PPL; u++) {
        const int32_t pt = first + u * kThreads < p.points ? first + u * kThreads : 0;
        c[u] = reinterpret_cast<const Coords<T, DIM>*>(wsn + p.lay.coords)[pt];
#pragma unroll
        for (int i = 0; i < NE; i++) {
            rank[u][i] = wsn[p.lay.ranks + (size_t)i * p.points + pt];
        }
    }
    uint32_t start[PPL][NE];
#pragma unroll
    for (int u = 0; u < PPL; u++) {
        for_entries<T, DIM, INTERP>(c[u], p, [&](int i, int32_t cell) {
            start[u][i] = wsn[p.lay.starts + (cell >= 0 ? cell : 0)];
        });
    }
    const uint32_t phase = (uint32_t)phase_of(n, p);
#pragma unroll
    for (int u = 0; u < PPL; u++) {
        const int32_t pt = first + u * kThreads;
#pragma unroll
        for (int i = 0; i < NE; i++) {
            if (pt < p.points && rank[u][i] != kNoRank) {
                wsn[p.lay.list + start[u][i] + rank[u][i]] = Mode<DIM, INTERP>::entry((uint32_t)pt + phase, (uint32_t)i);
            }
        }
    }
}

// Sorts one run (ascending entries, all distinct) into `out` with all threads of the workgroup: a bitmap of the entries
// that lie in a window of values, then every thread writes out the entries of its words behind those of the threads
// before it.  A run costs a pass over it per window of 32 * kBitWords values that it spans.
template <int kBitWords>
__device__ __forceinline__ void sort_run(const uint32_t* run, uint32_t len, uint32_t* out, uint32_t* bits,
                                         uint32_t* s_part)
{
    const int t = threadIdx.x;
    uint32_t lo = 0xFFFFFFFFu, hi = 0u;
    for (uint32_t i = t; i < len; i += kThreads) {
        const uint32_t v = run[i];
        lo = v < lo ? v : lo;
        hi = v > hi ? v : hi;
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        const uint32_t olo = __shfl_xor(lo, d), ohi = __shfl_xor(hi, d);
        lo = olo < lo ? olo : lo;
        hi = ohi > hi ? ohi : hi;
    }
    __syncthreads();  // the bitmap and s_part of the run before this one are done with
    if ((t & 63) == 0) {
        s_part[t >> 6] = lo;
        s_part[4 + (t >> 6)] = hi;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kThreads / 64; w++) {
        lo = s_part[w] < lo ? s_part[w] : lo;
        hi = s_part[4 + w] > hi ? s_part[4 + w] : hi;
    }
    uint32_t done = 0;
    while (done < len && lo <= hi) {  // lo: the first value of this window; every entry below it is written
        const uint32_t left = (hi - lo) / 32u + 1u;
        const uint32_t words = left < (uint32_t)kBitWords ? left : (uint32_t)kBitWords;
        const uint32_t each = (words + kThreads - 1u) / kThreads;
        for (uint32_t i = t; i < each * kThreads; i += kThreads) {
            bits[i] = 0u;
        }
        __syncthreads();
        for (uint32_t i = t; i < len; i += kThreads) {
            const uint32_t v = run[i] - lo;  // entries of earlier windows wrap round to huge values
            if (v < words * 32u) {
                atomicOr(&bits[v >> 5], 1u << (v & 31u));
            }
        }
        __syncthreads();
        uint32_t mine = 0;
        for (uint32_t i = 0; i < each; i++) {
            mine += (uint32_t)__builtin_popcount(bits[t * each + i]);
        }
        uint32_t incl = mine;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t up = __shfl_up(incl, d);
            incl += ((t & 63) >= d) ? up : 0u;
        }
        if ((t & 63) == 63) {
            s_part[t >> 6] = incl;
        }
        __syncthreads();
        uint32_t at = done + incl - mine;
        uint32_t total = 0;
#pragma unroll
        for (int w = 0; w < kThreads / 64; w++) {
            at += (w < (t >> 6)) ? s_part[w] : 0u;
            total += s_part[w];
        }
        for (uint32_t i = 0; i < each; i++) {
            uint32_t b = bits[t * each + i];
            while (b != 0u) {
                out[at++] = lo + (t * each + i) * 32u + (uint32_t)__builtin_ctz(b);
                b &= b - 1u;
            }
        }
        done += total;
        lo += words * 32u;
        __syncthreads();
    }
}

// The run (start, length) of each cell that element (x, y, z) is a corner of, in corner order.
template <int DIM, int INTERP>
__device__ __forceinline__ void runs_of(const uint32_t* __restrict__ wsn, const GatherParams& p, int32_t e, int32_t x,
                                        int32_t y, int32_t z, uint32_t* start, uint32_t* count)
{
    constexpr int R = Mode<DIM, INTERP>::kRuns;
    const uint32_t* starts = wsn + p.lay.starts;
    const uint32_t* counts = wsn + p.lay.counts;
    if constexpr (R == 1) {
        start[0] = starts[e];
        count[0] = counts[e];
    } else {
#pragma unroll
        for (int r = 0; r < R; r += 2) {
            const int ys = (r >> 1) & 1, zs = r >> 2;
            const int32_t row = (DIM == 3) ? (z + 1 - zs) * (p.H + 1) + (y + 1 - ys) : y + 1 - ys;
            const int32_t cell = row * (p.W + 1) + x;  // the cell of corner xs = 1; the next one is that of xs = 0
            uint2 s, c;
            __builtin_memcpy(&s, starts + cell, 8);
            __builtin_memcpy(&c, counts + cell, 8);
            start[r] = s.y;
            start[r + 1] = s.x;
            count[r] = c.y;
            count[r + 1] = c.x;
        }
    }
}

// LIST: contributions an element's list can hold (16 or 32).
template <typename T, int DIM, int INTERP, int CB, int LIST>
__global__ __launch_bounds__(kThreads) void gs_gather_kernel(const T* __restrict__ gout, T* __restrict__ dx,
                                                              uint32_t* __restrict__ ws, GatherParams p, uint32_t pieces,
                                                              uint32_t gather_blocks, uint32_t tiles,
                                                              int32_t chans_per_block, uint32_t sorters)
{
    typedef Mode<DIM, INTERP> M;
    constexpr int R = M::kRuns;
    constexpr int kBitWords = LIST * kThreads;  // the list memory, and the bitmap of a workgroup that sorts runs
    __shared__ uint32_t list[kBitWords];  // entry i of lane t at [i * kThreads + t]: a bank of its own
    __shared__ uint32_t s_part[2 * kThreads / 64];
    const int t = threadIdx.x;
    if (blockIdx.x >= gather_blocks) {
        // a spare workgroup: sorts long runs (of elements that the lanes below leave to the crowded kernel)
        const uint32_t i = blockIdx.x - gather_blocks;
        uint32_t* wsn = ws + (size_t)(i / sorters) * p.lay.item_words;
        const uint32_t runs = wsn[1];
        for (uint32_t r = i % sorters; r < runs; r += sorters) {
            const uint32_t cell = wsn[p.lay.runs + r];
            const uint32_t start = wsn[p.lay.starts + cell];
            sort_run<kBitWords>(wsn + p.lay.list + start, wsn[p.lay.counts + cell], wsn + p.lay.ranks + start, list, s_part);
        }
        return;
    }
    uint32_t n, local;
    if (!piece_of_block(blockIdx.x, pieces, pieces / (uint32_t)p.N, &n, &local)) {
        return;
    }
    uint32_t* wsn = ws + (size_t)n * p.lay.item_words;
    const uint32_t cblock = local / tiles;
    const int32_t e = (int32_t)((local - cblock * tiles) * kThreads + t);
    if (e >= p.elements) {
        return;
    }
    const int32_t x = e % p.W, yz = e / p.W;
    const int32_t y = (DIM == 3) ? yz % p.H : yz, z = (DIM == 3) ? yz / p.H : 0;
    uint32_t start[R], count[R], len = 0;
    runs_of<DIM, INTERP>(wsn, p, e, x, y, z, start, count);
#pragma unroll
    for (int r = 0; r < R; r++) {
        len += count[r];
    }
    if (len > (uint32_t)LIST) {
        if (cblock == 0) {
            wsn[p.lay.crowded + atomicAdd(&wsn[2], 1u)] = (uint32_t)e;
        }
        return;
    }
    uint32_t* mine = list + t;
    const uint32_t* entries = wsn + p.lay.list;
    // the first two entries of every run without a loop (as many as a smooth grid has)
    uint32_t first[R], second[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        first[r] = count[r] > 0u ? entries[start[r]] : 0u;
        second[r] = count[r] > 1u ? entries[start[r] + 1u] : 0u;
    }
    uint32_t at = 0;
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (count[r] > 0u) {
            mine[at * kThreads] = M::key(first[r], r);
        }
        if (count[r] > 1u) {
            mine[(at + 1u) * kThreads] = M::key(second[r], r);
        }
        for (uint32_t i = 2; i < count[r]; i++) {
            mine[(at + i) * kThreads] = M::key(entries[start[r] + i], r);
        }
        at += count[r];
    }
    if (__builtin_amdgcn_ballot_w64(len > 8u) == 0) {
        sort_list<8, kThreads>(mine, len);
    } else if (LIST <= 16 || __builtin_amdgcn_ballot_w64(len > 16u) == 0) {
        sort_list<16, kThreads>(mine, len);
    } else {
        sort_list<LIST, kThreads>(mine, len);
    }
    const Coords<T, DIM>* coords = reinterpret_cast<const Coords<T, DIM>*>(wsn + p.lay.coords);
    const uint32_t phase = (uint32_t)phase_of(n, p);
    const int32_t c_begin = (int32_t)cblock * chans_per_block;
    const int32_t c_end = (c_begin + chans_per_block < p.C) ? c_begin + chans_per_block : p.C;
    for (int32_t c0 = c_begin; c0 < c_end; c0 += CB) {
        const int32_t nc = (c_end - c0 < CB) ? c_end - c0 : CB;
        const T* go = gout + ((int64_t)n * p.C + c0) * (int64_t)p.points;
        float acc[CB];
#pragma unroll
        for (int j = 0; j < CB; j++) {
            acc[j] = 0.0f;
        }
        // two entries in flight: the operands of the entry after this one are asked for before this one is folded in
        struct Operands {
            Coords<T, DIM> at;
            uint32_t tap;
            T go[CB];
        };
        auto fetch = [&](uint32_t i, Operands& o) {
            const uint32_t key = mine[i * kThreads];
            const uint32_t pt = M::q_of(key) - phase;
            o.tap = M::tap_of(key);
            if (INTERP != 1) {
                o.at = coords[pt];
            }
#pragma unroll
            for (int j = 0; j < CB; j++) {
                if (j < nc) {
                    o.go[j] = go[(int64_t)j * p.points + pt];
                }
            }
        };
        auto fold = [&](const Operands& o) {
            const float w = weight_of<T, DIM, INTERP>(o.at, o.tap, x, y, z);
#pragma unroll
            for (int j = 0; j < CB; j++) {
                acc[j] = rt<T>(acc[j] + value_of<T, INTERP>(ElemIO<T>::load(&o.go[j]), w));
            }
        };
        Operands a{}, b{};
        if (len > 0u) {
            const uint32_t last = len - 1u;
            fetch(0u, a);
            for (uint32_t i = 0; i < len; i += 2) {
                fetch(i + 1u < len ? i + 1u : last, b);
                fold(a);
                fetch(i + 2u < len ? i + 2u : last, a);
                if (i + 1u < len) {
                    fold(b);
                }
            }
        }
#pragma unroll
        for (int j = 0; j < CB; j++) {
            if (j < nc) {
                store_streaming<T>(dx + ((int64_t)n * p.C + c0 + j) * (int64_t)p.elements + e, acc[j]);
            }
        }
    }
}

// Elements with more contributions than the gather kernel takes: a wavefront per element and 64 channels.
template <typename T, int DIM, int INTERP>
__global__ __launch_bounds__(kThreads) void gs_gather_crowded_kernel(const T* __restrict__ gout, T* __restrict__ dx,
                                                                      const uint32_t* __restrict__ ws, GatherParams p)
{
    typedef Mode<DIM, INTERP> M;
    constexpr int R = M::kRuns;
    constexpr int kWaves = kThreads / 64;
    __shared__ uint32_t s_window[kWaves][R][64];      // short runs, sorted
    __shared__ uint32_t s_key[kWaves][kCountedMost];  // keys in order: the next 64, or all
    __shared__ __align__(16) float s_val[kWaves][kFoldChans][kFoldPitch];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t n = blockIdx.y;
    const uint32_t* wsn = ws + (size_t)n * p.lay.item_words;
    const uint32_t chan_blocks = (uint32_t)(p.C + 63) / 64u;
    const uint32_t jobs = wsn[2] * chan_blocks;
    const uint32_t phase = (uint32_t)phase_of(n, p);
    const Coords<T, DIM>* coords = reinterpret_cast<const Coords<T, DIM>*>(wsn + p.lay.coords);
    uint32_t(*window)[64] = s_window[wave];
    uint32_t* keys = s_key[wave];
    float(*val)[kFoldPitch] = s_val[wave];
    // the wavefronts of a workgroup share nothing: what a wavefront writes to LDS it reads back itself, in order
    auto landed = [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); __builtin_amdgcn_wave_barrier(); };
    for (uint32_t job = blockIdx.x * kWaves + wave; job < jobs; job += gridDim.x * kWaves) {
        const int32_t e = (int32_t)wsn[p.lay.crowded + job / chan_blocks];
        const int32_t c_first = (int32_t)(job % chan_blocks) * 64;
        const int32_t nc = (p.C - c_first < 64) ? p.C - c_first : 64;
        const int32_t x = e % p.W, yz = e / p.W;
        const int32_t y = (DIM == 3) ? yz % p.H : yz, z = (DIM == 3) ? yz / p.H : 0;
        uint32_t start[R], left[R];
        runs_of<DIM, INTERP>(wsn, p, e, x, y, z, start, left);
        uint32_t total = 0;
        const uint32_t* from[R];  // where the rest of a run is read from
        bool whole[R];            // the run is short: sorted here, once, and kept
        uint32_t skip[R];         // entries of a short run already taken
#pragma unroll
        for (int r = 0; r < R; r++) {
            start[r] = (uint32_t)__builtin_amdgcn_readfirstlane((int)start[r]);
            left[r] = (uint32_t)__builtin_amdgcn_readfirstlane((int)left[r]);
            total += left[r];
            whole[r] = left[r] <= kSortedRun;
            skip[r] = 0u;
            from[r] = wsn + (whole[r] ? p.lay.list : p.lay.ranks) + start[r];
        }
        const bool counted = R > 1 && total <= kCountedMost;
        if (counted) {
            // a key or two a lane, whose place is the number of lesser ones
            constexpr int kRegs = (int)(kCountedMost / 64u);
            uint32_t own[kRegs], rank[kRegs];
#pragma unroll
            for (int m = 0; m < kRegs; m++) {
                const uint32_t i = (uint32_t)(m * 64 + lane);
                uint32_t before = 0, run = 0, at = 0;
#pragma unroll
                for (int r = 0; r < R; r++) {
                    if (i >= before) {
                        run = (uint32_t)r;
                        at = (uint32_t)(from[r] - wsn) + i - before;
                    }
                    before += left[r];
                }
                own[m] = (i < total) ? M::key(wsn[at], run) : 0xFFFFFFFFu;
                rank[m] = 0u;
            }
#pragma unroll
            for (int m = 0; m < kRegs; m++) {
                const uint32_t most = total > (uint32_t)(m * 64) ? total - (uint32_t)(m * 64) : 0u;
                const uint32_t here = most < 64u ? most : 64u;
                for (uint32_t j = 0; j < here; j += 8u) {
#pragma unroll
                    for (uint32_t u = 0; u < 8u; u++) {
                        const uint32_t other = (uint32_t)__builtin_amdgcn_readlane((int)own[m], (int)(j + u));
#pragma unroll
                        for (int q = 0; q < kRegs; q++) {
                            rank[q] += (other < own[q]) ? 1u : 0u;
                        }
                    }
                }
            }
#pragma unroll
            for (int m = 0; m < kRegs; m++) {
                if ((uint32_t)(m * 64 + lane) < total) {
                    keys[rank[m]] = own[m];
                }
            }
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (!counted && whole[r] && left[r] > 0u) {
                const bool have = (uint32_t)lane < left[r];
                const uint32_t v = have ? from[r][lane] : 0xFFFFFFFFu;
                uint32_t rank = 0;
                for (uint32_t i = 0; i < left[r]; i++) {
                    const uint32_t other = (uint32_t)__shfl((int)v, (int)i);
                    rank += (other < v) ? 1u : 0u;
                }
                if (have) {
                    window[r][rank] = v;
                }
            }
        }
        landed();
        uint32_t ahead[R];  // the next 64 entries of the long runs
        auto look_ahead = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < R; r++) {
                ahead[r] = 0xFFFFFFFFu;
                if (!counted && !whole[r] && (uint32_t)lane < left[r]) {
                    ahead[r] = from[r][lane];
                }
            }
        };
        look_ahead();
        uint32_t taken_before = 0;  // of the keys
        float acc = 0.0f;           // of channel c_first + lane
        while (total > 0u) {
            const uint32_t batch = total < 64u ? total : 64u;
            if (!counted) {
                // the next entries of every run, and behind a run's last one an entry beyond all
                uint32_t mine[R], held[R], rank[R];
#pragma unroll
                for (int r = 0; r < R; r++) {
                    held[r] = left[r] < 64u ? left[r] : 64u;
                    mine[r] = ahead[r];
                    if (whole[r] && (uint32_t)lane < held[r]) {
                        mine[r] = window[r][skip[r] + lane];
                    }
                    rank[r] = (uint32_t)lane;
                }
                // the rank of every one of them among all: entries of another run come first when their chunk is earlier, or the
                // same and their corner's number lower
#pragma unroll
                for (int r = 0; r < R; r++) {
#pragma unroll
                    for (int o = 0; o < r; o++) {
                        if (held[r] > 0u && held[o] > 0u) {
                            const uint32_t longest = held[r] > held[o] ? held[r] : held[o];
                            // how many of run o lie before this lane's entry of run r, and of run r before its entry of run o
                            const uint32_t in_r = mine[r] >> 8, in_o = mine[o] >> 8;
                            uint32_t less_o = 0, less_r = 0;
#pragma unroll
                            for (uint32_t d = 32; d > 0u; d >>= 1) {
                                if (d > longest) {
                                    continue;
                                }
                                const uint32_t chunk_o = (uint32_t)__shfl((int)in_o, (int)(less_o + d - 1u));
                                const uint32_t chunk_r = (uint32_t)__shfl((int)in_r, (int)(less_r + d - 1u));
                                less_o += (chunk_o <= in_r) ? d : 0u;
                                less_r += (chunk_r < in_o) ? d : 0u;
                            }
                            if (longest == 64u) {  // the last one
                                less_o += ((uint32_t)__shfl((int)in_o, (int)less_o) <= in_r) ? 1u : 0u;
                                less_r += ((uint32_t)__shfl((int)in_r, (int)less_r) < in_o) ? 1u : 0u;
                            }
                            rank[r] += less_o;
                            rank[o] += less_r;
                        }
                    }
                }
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const bool take = (uint32_t)lane < held[r] && rank[r] < batch;
                    if (take) {
                        keys[rank[r]] = M::key(mine[r], r);
                    }
                    const uint32_t taken = (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(take));
                    left[r] -= taken;
                    if (whole[r]) {
                        skip[r] += taken;
                    } else {
                        from[r] += taken;
                    }
                }
                look_ahead();
            }
            total -= batch;
            landed();
            const uint32_t key = keys[taken_before + ((uint32_t)lane < batch ? (uint32_t)lane : 0u)];
            taken_before += counted ? batch : 0u;
            const uint32_t pt = M::q_of(key) - phase;
            const float w = weight_of<T, DIM, INTERP>(coords[pt], M::tap_of(key), x, y, z);
            const T* go = gout + (n * p.C + c_first) * (int64_t)p.points + pt;
            T got[kFoldChans];  // of the next channels
            auto fetch = [&](int32_t g) __attribute__((always_inline)) {
#pragma unroll
                for (int j = 0; j < kFoldChans; j++) {
                    if (g + j < nc) {
                        got[j] = go[(int64_t)(g + j) * p.points];
                    }
                }
            };
            fetch(0);
            for (int32_t g = 0; g < nc; g += kFoldChans) {
                landed();
#pragma unroll
                for (int j = 0; j < kFoldChans; j++) {
                    if (g + j < nc) {
                        val[j][lane] = ((uint32_t)lane < batch) ? value_of<T, INTERP>(ElemIO<T>::load(&got[j]), w) : 0.0f;
                    }
                }
                fetch(g + kFoldChans);
                landed();
                if (lane >= g && lane < g + kFoldChans && lane < nc) {
                    acc = add_in_order<T>(acc, val[lane - g], batch);
                }
            }
            landed();
        }
        if (lane < nc) {
            store_streaming<T>(dx + (n * p.C + c_first + lane) * (int64_t)p.elements + e, acc);
        }
    }
}

inline uint32_t swizzled_blocks(int64_t pieces) { return (uint32_t)((pieces + 7) / 8 * 8); }

template <typename T, int DIM, int INTERP, int CB, int LIST>
hipError_t launch_gather(const GradGatherArgs& a, const GatherPlan& pl, hipStream_t stream)
{
    const uint32_t pieces = (uint32_t)a.N * pl.tiles * pl.cblocks;
    const uint32_t blocks = swizzled_blocks(pieces);
    // workgroups that sort long runs: a turn of the chip at most, and none an item could not use
    const int64_t most_runs = a.points * Mode<DIM, INTERP>::kEntries / (kSortedRun + 1);
    int64_t sorters = 512 / a.N > 0 ? 512 / a.N : 1;
    sorters = sorters < most_runs ? sorters : most_runs;
    hipLaunchKernelGGL((gs_gather_kernel<T, DIM, INTERP, CB, LIST>), dim3(blocks + (uint32_t)(sorters * a.N)), dim3(kThreads), 0,
                       stream, (const T*)a.gout, (T*)a.dx, (uint32_t*)a.scratch, pl.p, pieces, blocks, pl.tiles,
                       pl.chans_per_block, (uint32_t)(sorters > 0 ? sorters : 1));
    return hipGetLastError();
}

template <typename T, int DIM, int INTERP>
hipError_t run_mode(const GradGatherArgs& a, const GatherPlan& pl, hipStream_t stream)
{
    const GatherParams& p = pl.p;
    uint32_t* ws = (uint32_t*)a.scratch;
    const uint32_t clear_words = p.lay.starts;
    hipLaunchKernelGGL(gs_gather_clear_kernel, dim3((clear_words / 4 + kThreads - 1) / kThreads, (unsigned)a.N),
                       dim3(kThreads), 0, stream, ws, clear_words, p.lay.item_words);
    constexpr int kPoints = kThreads * points_per_lane<DIM, INTERP>();
    const uint32_t per_item = (uint32_t)((a.points + kPoints - 1) / kPoints);
    const uint32_t pieces = (uint32_t)a.N * per_item;
    hipLaunchKernelGGL((gs_gather_count_kernel<T, DIM, INTERP>), dim3(swizzled_blocks(pieces)), dim3(kThreads), 0, stream,
                       (const T*)a.grid, ws, p, pieces, per_item);
    hipLaunchKernelGGL(gs_gather_place_kernel,
                       dim3((unsigned)((p.cells + kPlaceThreads * kPlaceCells - 1) / (kPlaceThreads * kPlaceCells)),
                            (unsigned)a.N),
                       dim3(kPlaceThreads), 0, stream, ws, p);
    hipLaunchKernelGGL((gs_gather_fill_kernel<T, DIM, INTERP>), dim3(swizzled_blocks(pieces)), dim3(kThreads), 0, stream, ws,
                       p, pieces, per_item);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        return e;
    }
    switch (pl.cb * 64 + pl.list) {
        case 1 * 64 + 16: e = launch_gather<T, DIM, INTERP, 1, 16>(a, pl, stream); break;
        case 2 * 64 + 16: e = launch_gather<T, DIM, INTERP, 2, 16>(a, pl, stream); break;
        case 4 * 64 + 16: e = launch_gather<T, DIM, INTERP, 4, 16>(a, pl, stream); break;
        case 8 * 64 + 16: e = launch_gather<T, DIM, INTERP, 8, 16>(a, pl, stream); break;
        case 1 * 64 + 32: e = launch_gather<T, DIM, INTERP, 1, 32>(a, pl, stream); break;
        case 2 * 64 + 32: e = launch_gather<T, DIM, INTERP, 2, 32>(a, pl, stream); break;
        case 4 * 64 + 32: e = launch_gather<T, DIM, INTERP, 4, 32>(a, pl, stream); break;
        default: e = launch_gather<T, DIM, INTERP, 8, 32>(a, pl, stream); break;
    }
    if (e != hipSuccess) {
        return e;
    }
    const int64_t most = a.points * Mode<DIM, INTERP>::kEntries * Mode<DIM, INTERP>::kRuns / (pl.list + 1);
    if (most > 0) {  // else no element can be crowded
        const int64_t per = 1024 / a.N > 1 ? 1024 / a.N : 1;
        hipLaunchKernelGGL((gs_gather_crowded_kernel<T, DIM, INTERP>), dim3((unsigned)per, (unsigned)a.N), dim3(kThreads),
                           0, stream, (const T*)a.gout, (T*)a.dx, ws, p);
    }
    return hipGetLastError();
}

template <typename T>
hipError_t run_typed(const GradGatherArgs& a, const GatherPlan& pl, hipStream_t stream)
{
    switch (a.dim * 4 + a.interp) {
        case 2 * 4 + 0: return run_mode<T, 2, 0>(a, pl, stream);
        case 2 * 4 + 1: return run_mode<T, 2, 1>(a, pl, stream);
        case 2 * 4 + 2: return run_mode<T, 2, 2>(a, pl, stream);
        case 3 * 4 + 0: return run_mode<T, 3, 0>(a, pl, stream);
        case 3 * 4 + 1: return run_mode<T, 3, 1>(a, pl, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

int64_t grad_gather_words(const GradGatherArgs& a)
{
    if (const int64_t words = grad_tiles_words(a); words > 0) {
        return words;
    }
    const GatherPlan pl = gather_plan(a);
    return pl.ok ? (int64_t)pl.p.lay.item_words * pl.group : 0;
}

hipError_t run_grad_gather(const GradGatherArgs& a, hipStream_t stream, bool* dgrid_done)
{
    if (grad_tiles_words(a) > 0) {
        return run_grad_tiles(a, stream, dgrid_done);
    }
    GatherPlan pl = gather_plan(a);
    if (!pl.ok || a.dx == nullptr || a.gout == nullptr || a.grid == nullptr || a.scratch == nullptr) {
        return hipErrorInvalidValue;
    }
    // the items are independent: a group of them after the other, each in all of the scratch
    const int64_t esz = elem_size(a.elem);
    for (int64_t first = 0; first < a.N; first += pl.group) {
        GradGatherArgs g = a;
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
    return hipSuccess;
}

}  // namespace opscv
