// What the kernels of the input gradient by tiles share (gs_grad_tiles.hip, gs_grad_tiles_crowded.hip): scans, the cell of a
// point, a tile's segments, weights in LDS.
#pragma once

#include <hip/hip_runtime.h>

#include "gs_grad_points.hpp"
#include "gs_grad_tiles_plan.hpp"

namespace opscv {

// the tiles on the list, after the gather kernel (gs_grad_tiles_crowded.hip)
hipError_t run_crowded_tiles(const GradGatherArgs& a, const TilesPlan& pl, hipStream_t stream);

__device__ __forceinline__ void landed()
{
    // what a wavefront writes to LDS it reads back itself, in order
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ uint32_t bits_below(uint64_t mask)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// Inclusive sum over the wavefront: within rows of 16 lanes, then from row to row.
__device__ __forceinline__ uint32_t wave_scan(uint32_t v)
{
    int s = (int)v;
    s += __builtin_amdgcn_update_dpp(0, s, 0x111, 0xf, 0xf, false);  // row_shr:1
    s += __builtin_amdgcn_update_dpp(0, s, 0x112, 0xf, 0xf, false);
    s += __builtin_amdgcn_update_dpp(0, s, 0x114, 0xf, 0xf, false);
    s += __builtin_amdgcn_update_dpp(0, s, 0x118, 0xf, 0xf, false);
    s += __builtin_amdgcn_update_dpp(0, s, 0x142, 0xa, 0xf, false);  // row_bcast:15 to rows 1 and 3
    s += __builtin_amdgcn_update_dpp(0, s, 0x143, 0xc, 0xf, false);  // row_bcast:31 to rows 2 and 3
    return (uint32_t)s;
}

// The cell of a point: the lattice of low corners for linear interpolation, the element for nearest.  False: no corner
// is inside (or the coordinate is not a number; sizes are exact in single precision: launch plan).
template <typename T, int DIM, int INTERP>
__device__ __forceinline__ bool low_corner(const Coords<T, DIM>& c, const TilesParams& p, int32_t* x, int32_t* y, int32_t* z)
{
    constexpr float least = (INTERP == 1) ? 0.0f : -1.0f;
    auto axis = [&](int i, int32_t size, int32_t* cell) {
        const float v = ElemIO<T>::load(&c.v[i]);
        const float f = (INTERP == 1) ? __builtin_rintf(v) : __builtin_floorf(v);
        const bool in = f >= least && f < (float)size;
        *cell = (int32_t)(in ? f : 0.0f);
        return in;
    };
    bool in = axis(0, p.W, x);
    in = axis(1, p.H, y) && in;
    *z = 0;
    if constexpr (DIM == 3) {
        in = axis(2, p.D, z) && in;
    }
    return in;
}

// Sums of the wavefronts before this one, and of all, from every wavefront's in LDS.
template <int WAVES>
__device__ __forceinline__ uint32_t sums_before(const uint32_t* s_scan, int wave, int lane, uint32_t* all)
{
    const uint32_t incl = wave_scan(lane < WAVES ? s_scan[lane < WAVES ? lane : 0] : 0u);
    *all = (uint32_t)__builtin_amdgcn_readlane((int)incl, WAVES - 1);
    return wave > 0 ? (uint32_t)__builtin_amdgcn_readlane((int)incl, wave - 1) : 0u;
}

// A tile's segments that are not empty, by a workgroup of TH lanes: points before each (and behind the last all of them), and
// block << 14 | first record.  Packed sums: segments above 21 bits of points; both fit by launch plan.
template <int TH>
__device__ __forceinline__ void tile_segments(const uint32_t* __restrict__ item, const TilesParams& p, uint32_t tile,
                                              uint32_t* s_before, uint32_t* s_where, uint32_t* s_scan, uint32_t* segments,
                                              uint32_t* points)
{
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    uint32_t segs = 0, total = 0;
    for (int32_t b0 = 0; b0 < p.blocks; b0 += TH) {
        const int32_t b = b0 + t;
        const uint32_t w = (b < p.blocks) ? item[p.lay.segments + (size_t)b * p.tiles + tile] : 0u;
        const uint32_t count = w >> 16, packed = count | (count > 0u ? 1u << 21 : 0u);
        uint32_t incl = 0u;
        if (b0 + wave * 64 < p.blocks) {
            incl = wave_scan(packed);
        }
        if (lane == 63) {
            s_scan[wave] = incl;
        }
        __syncthreads();
        uint32_t all;
        const uint32_t before = sums_before<TH / 64>(s_scan, wave, lane, &all) + incl - packed;
        if (count > 0u) {
            const uint32_t at = segs + (before >> 21);
            s_before[at] = total + (before & 0x1FFFFFu);
            s_where[at] = ((uint32_t)b << 14) | (w & 0xFFFFu);
        }
        segs += all >> 21;
        total += all & 0x1FFFFFu;
        __syncthreads();
    }
    if (t == 0) {
        s_before[segs] = total;
    }
    *segments = segs;
    *points = total;
}

// Weights of the points in LDS, plane by plane (a lane reads a weight of some point: neighbours in a plane lie in different
// banks): every corner's, values of the element type; of volumes in single precision, which would fill LDS, the products
// of the four corners along x and y and the two distances along z.  The last of a plane is zero.
template <typename T, int DIM, int CAP>
struct Weights {
    static constexpr bool kProducts = DIM == 3 && sizeof(T) == 4;
    static constexpr int kPlanes = kProducts ? 6 : (1 << DIM);
    static constexpr uint32_t kStride = CAP + 1;
    T v[kPlanes * kStride];
    __device__ __forceinline__ void put(uint32_t i, const Coords<T, DIM>& c)
    {
        float d[DIM][2];  // to the high edge and from the low edge of the cell, as the decisions of the taps have them
#pragma unroll
        for (int k = 0; k < DIM; k++) {
            const float f = ElemIO<T>::load(&c.v[k]), low = __builtin_floorf(f);
            d[k][0] = (low + 1.0f) - f;
            d[k][1] = f - low;
        }
#pragma unroll
        for (int k = 0; k < kPlanes; k++) {
            float w;
            if constexpr (kProducts) {
                w = (k < 4) ? d[0][k & 1] * d[1][(k >> 1) & 1] : d[DIM - 1][k & 1];
            } else {
                w = d[0][k & 1] * d[1][(k >> 1) & 1];
                if constexpr (DIM == 3) {
                    w = w * d[DIM - 1][k >> 2];
                }
            }
            ElemIO<T>::store(&v[k * kStride + i], as_fp32_value(w));
        }
    }
    __device__ __forceinline__ float get(uint32_t i, uint32_t tap) const
    {
        if constexpr (kProducts) {
            return v[(tap & 3u) * kStride + i] * v[((tap >> 2) + 4u) * kStride + i];
        } else {
            return ElemIO<T>::load(&v[tap * kStride + i]);
        }
    }
    __device__ __forceinline__ void clear_last(int t)
    {
        if (t < kPlanes) {
            ElemIO<T>::store(&v[t * kStride + CAP], 0.0f);
        }
    }
};

}  // namespace opscv
