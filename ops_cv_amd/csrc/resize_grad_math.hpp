// Which elements of the incoming gradient an element of the resize gradient visits, and their sum: what the kernels of
// resize_grad.hip and resize_grad_rows.hip share.
#pragma once

#include <hip/hip_runtime.h>

#include "resize_grad_plan.hpp"
#include "sampler_math.hpp"

namespace opscv {

// resize_grad_rows.hip
hipError_t run_resize_grad_rows(const ResizeGradArgs& a, const RowsPlan& p, hipStream_t stream);

// The visiting loops of resize_grad_kernel over a row-major array whose element (y0, x0) is base[0].
template <typename TI>
__device__ __forceinline__ float visit_sum(const TI* base, int32_t pitch, int32_t y0, int32_t x0, int32_t in_y_start,
                                           int32_t in_x_start, float out_y_start, float out_x_start, float fh,
                                           float fw, float scale_h, float scale_w, float last_y, float last_x,
                                           int32_t Hd, int32_t Wd, int32_t ci = 1, int32_t ch = 0)
{
    // ci, ch: channels-last rows hold ci elements per pixel, this lane's channel is ch (x0 counts elements)
    float acc = 0.0f;
    float out_y = out_y_start;
    for (int32_t in_y = in_y_start; out_y < fh + 1.0f && in_y < Hd; in_y++) {
        const float yc = __builtin_fmaxf(0.0f, __builtin_fminf(out_y, last_y));
        const float y_lerp = 1.0f - __builtin_fabsf(yc - fh);
        const TI* row = base + (int64_t)(in_y - y0) * pitch;
        float out_x = out_x_start;
        for (int32_t in_x = in_x_start; out_x < fw + 1.0f && in_x < Wd; in_x++) {
            const float xc = __builtin_fmaxf(0.0f, __builtin_fminf(out_x, last_x));
            const float x_lerp = 1.0f - __builtin_fabsf(xc - fw);
            acc += ElemIO<TI>::load(row + ((int64_t)in_x * ci + ch - x0)) * y_lerp * x_lerp;
            out_x += scale_w;
        }
        out_y += scale_h;
    }
    return acc;
}

// offset: half a pixel or none
__device__ __forceinline__ int32_t first_visited(int32_t i, float inv_scale, int32_t len_dst, float offset)
{
    const float f = __builtin_ceilf(((float)i - 1.0f + offset) * inv_scale - offset);
    // a start at or beyond the end visits nothing, whatever its exact value
    return (f > 0.0f) ? ((f < (float)len_dst) ? (int32_t)f : len_dst) : 0;
}

template <bool HALF_PIXEL>
__device__ __forceinline__ int32_t first_visited(int32_t i, float inv_scale, int32_t len_dst)
{
    return first_visited(i, inv_scale, len_dst, HALF_PIXEL ? 0.5f : 0.0f);
}

}  // namespace opscv
