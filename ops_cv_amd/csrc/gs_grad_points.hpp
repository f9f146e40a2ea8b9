// Grid points of the samplers' backward as the kernels of the input gradient see them (gs_grad_gather.hip,
// gs_grad_tiles.hip): source coordinates, the weight of a contribution and what it adds, and the chunks of the order.
#pragma once

#include <hip/hip_runtime.h>

#include "fast_div.hpp"
#include "gs2d_grad_math.hpp"
#include "gs3d_grad_math.hpp"

namespace opscv {

// source coordinates of a point: values of the element type
template <typename T, int DIM>
struct Coords {
    T v[DIM == 3 ? 4 : 2];
};

template <typename P>
__device__ __forceinline__ int32_t phase_of(int64_t n, const P& p)
{
    return (int32_t)((((p.first_item + n) % p.items_per_core) * (int64_t)p.points) % kChunkPoints3);
}

// The source coordinates of a grid point, as the tap decisions of gs2d_grad_math.hpp and gs3d_grad_math.hpp form them
// (values of the element type).
template <typename T, int DIM, int INTERP, typename P>
__device__ __forceinline__ Coords<T, DIM> coords_of(const T* __restrict__ g, const P& p)
{
    Coords<T, DIM> c;
    float m;
    auto axis = [&](int i, int32_t size) {
        const float v = ElemIO<T>::load(g + i);
        float f;
        if (INTERP == 2) {
            f = unnormalize_set_grad<T>(v, size, p.align, &m);
        } else if (p.pad == 2) {
            // the size passes an asm statement, so that what a reflection needs of it (conversions, a reciprocal for the
            // remainder: 120 instructions) is not worked out ahead by every wavefront of the other paddings too
            int32_t reflected = size;
            asm volatile("" : "+s"(reflected));
            f = source_index_set_grad<T>(v, reflected, 2, p.align, &m);
        } else {
            f = source_index_set_grad<T>(v, size, p.pad == 1 ? 1 : 0, p.align, &m);
        }
        ElemIO<T>::store(&c.v[i], f);
    };
    axis(0, p.W);
    axis(1, p.H);
    if constexpr (DIM == 3) {
        axis(2, p.D);
        c.v[3] = c.v[2];
    }
    return c;
}

// The weight of a contribution (unused for nearest): the products of gs2d_grad_math.hpp / gs3d_grad_math.hpp.
template <typename T, int DIM, int INTERP>
__device__ __forceinline__ float weight_of(const Coords<T, DIM>& c, uint32_t tap, int32_t x, int32_t y, int32_t z)
{
    const float fx = ElemIO<T>::load(&c.v[0]), fy = ElemIO<T>::load(&c.v[1]);
    if constexpr (INTERP == 1) {
        return 1.0f;
    } else if constexpr (INTERP == 2) {
        auto coefficient = [](uint32_t i, float t) {
            // the i-th of cubic_coefficients()
            const float u = (i >= 2) ? 1.0f - t : t;
            const float outer = cubic_convolution2((i == 0) ? t + 1.0f : 2.0f - t, -0.75f);
            const float inner = cubic_convolution1(u, -0.75f);
            return (i == 0 || i == 3) ? outer : inner;
        };
        return coefficient(tap >> 2, fx - __builtin_floorf(fx)) * coefficient(tap & 3u, fy - __builtin_floorf(fy));
    } else {
        // corner (xs, ys, zs) of the cell is element (x, y, z): the low corner is that much below it
        const bool xs = tap & 1u, ys = tap & 2u, zs = tap & 4u;
        const float wx = xs ? fx - (float)(x - 1) : (float)(x + 1) - fx;
        const float wy = ys ? fy - (float)(y - 1) : (float)(y + 1) - fy;
        if constexpr (DIM == 3) {
            const float fz = ElemIO<T>::load(&c.v[2]);
            const float wz = zs ? fz - (float)(z - 1) : (float)(z + 1) - fz;
            return rt<T>(as_fp32_value(wx * wy * wz));
        } else {
            return rt<T>(as_fp32_value(wx * wy));
        }
    }
}

// One more contribution, added with the reference's roundings (contribution() of gs2d_grad.hip, contribution3()).
template <typename T, int INTERP>
__device__ __forceinline__ float value_of(float go, float w)
{
    return (INTERP == 1) ? rt<T>(go) : rt<T>(as_fp32_value(w * go));
}

// A crowded element's sum goes on over `count` of 64 contributions in LDS (on the 16-byte grid, zeros behind the last: they change
// no sum that started at +0), a chain of additions: its operands are loaded 16 ahead, so that it never waits for LDS.
template <typename T>
__device__ __forceinline__ float add_in_order(float sum, const float* values, uint32_t count)
{
    float4 a[4], b[4];
    auto load = [&](float4 (&v)[4], int at) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            v[i] = *reinterpret_cast<const float4*>(values + at + 4 * i);
        }
    };
    auto add = [&](const float4 (&v)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            sum = rt<T>(sum + v[i].x);
            sum = rt<T>(sum + v[i].y);
            sum = rt<T>(sum + v[i].z);
            sum = rt<T>(sum + v[i].w);
        }
    };
    load(a, 0);
    load(b, 16);
    add(a);
    if (count > 16u) {
        load(a, 32);
        add(b);
        if (count > 32u) {
            load(b, 48);
            add(a);
            if (count > 48u) {
                add(b);
            }
        }
    }
    return sum;
}

// Work of a launch cut into `per_item` pieces per batch item, dealt out so that neighbouring pieces run on one XCD
// (workgroups go to the eight XCDs in turn): XCD k takes the k-th eighth of all pieces.  Pieces beyond the last: false.
__device__ __forceinline__ bool piece_of_block(uint32_t block, uint32_t pieces, uint32_t* piece)
{
    const uint32_t per_xcd = (pieces + 7u) >> 3;
    *piece = (block & 7u) * per_xcd + (block >> 3);
    return (block >> 3) < per_xcd && *piece < pieces;
}

__device__ __forceinline__ bool piece_of_block(uint32_t block, uint32_t pieces, uint32_t per_item, uint32_t* n,
                                               uint32_t* local)
{
    uint32_t piece;
    const bool have = piece_of_block(block, pieces, &piece);
    *n = piece / per_item;
    *local = piece - *n * per_item;
    return have;
}

__device__ __forceinline__ bool piece_of_block(uint32_t block, uint32_t pieces, const FastDiv& per_item, uint32_t* n,
                                               uint32_t* local)
{
    uint32_t piece;
    const bool have = piece_of_block(block, pieces, &piece);
    *n = fast_div(piece, per_item);
    *local = piece - *n * per_item.div;
    return have;
}

}  // namespace opscv
