// Backward of the bilinear resize for gfx950, deterministic gather formulation.
//
// Replaces the reference device kernel
// image/resize_bilinear_v2_grad/op_kernel/arch35/resize_bilinear_v2_grad_simt_determine.h:56-117 and the scale rules
// of image/resize_bilinear_v2_grad/op_host/arch35/resize_bilinear_v2_grad_tiling_arch35.cpp:352-394.
//
// One lane per element (n, c, H, W) of the outgoing gradient.  It visits the incoming-gradient rows inY whose
// source coordinate outY = (inY + o) * scale - o lies in (H - 1, H + 1), starting at
// ceil((H - 1 + o) / scale - o) and advancing outY by repeated addition of the scale (as the reference does, so
// the rounding of every coordinate is the same), and likewise the columns; each visited element contributes
// g * (1 - |clamp(outY) - H|) * (1 - |clamp(outX) - W|), summed in fp32 in row-major visiting order.  No atomics:
// the result does not depend on scheduling.  The translation unit is compiled with -ffp-contract=off.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <type_traits>

#include "kernels.hpp"
#include "resize_grad_math.hpp"
#include "resize_grad_plan.hpp"
#include "sampler_math.hpp"

namespace opscv {

namespace {

// User-scale template (resize_bilinear_v2_grad_simt_determine_scales.h:77-305), for scales that are not the ratio
// of the sizes.  Same walk, but the source coordinate of every visited row/column is recomputed as
// scale * (i + o) - o instead of accumulated, and an element on the first or last row (column) of the outgoing
// gradient scans the incoming rows (columns) to the end and takes, per visited element, the weights of the taps
// that land on it (floor tap: 1 - |c - H|; next tap: c - floor(c)).
template <typename TI, typename TO, bool HALF_PIXEL, bool NHWC>
__global__ __launch_bounds__(kGradThreads) void resize_grad_scales_kernel(const TI* __restrict__ g, TO* __restrict__ y,
                                                                           int64_t total, int32_t C, int32_t Hs,
                                                                           int32_t Ws, int32_t Hd, int32_t Wd,
                                                                           float scale_h, float scale_w,
                                                                           float inv_scale_h, float inv_scale_w)
{
    const int64_t stride = (int64_t)gridDim.x * kGradThreads;
    const float offset = HALF_PIXEL ? 0.5f : 0.0f;
    const float last_y = (float)Hs - 1.0f, last_x = (float)Ws - 1.0f;
    auto source_index = [](float scale, int64_t i) {
        return HALF_PIXEL ? scale * ((float)i + 0.5f) - 0.5f : scale * (float)i;
    };
    for (int64_t idx = (int64_t)blockIdx.x * kGradThreads + threadIdx.x; idx < total; idx += stride) {
        int64_t t = idx;
        int32_t c, W, H;
        if (NHWC) {
            c = (int32_t)(t % C);
            t /= C;
            W = (int32_t)(t % Ws);
            t /= Ws;
            H = (int32_t)(t % Hs);
            t /= Hs;
        } else {
            W = (int32_t)(t % Ws);
            t /= Ws;
            H = (int32_t)(t % Hs);
            t /= Hs;
            c = (int32_t)(t % C);
            t /= C;
        }
        const int64_t n = t;
        const float fy0 = __builtin_ceilf(((float)H - 1.0f + offset) * inv_scale_h - offset);
        const float fx0 = __builtin_ceilf(((float)W - 1.0f + offset) * inv_scale_w - offset);
        const int64_t in_y_start = (fy0 > 0.0f) ? (int64_t)fy0 : 0;
        const int64_t in_x_start = (fx0 > 0.0f) ? (int64_t)fx0 : 0;
        const float out_y_start = ((float)in_y_start + offset) * scale_h - offset;
        const float out_x_start = ((float)in_x_start + offset) * scale_w - offset;
        const float fh = (float)H, fw = (float)W;
        const bool hb = (H == 0 || H == Hs - 1), wb = (W == 0 || W == Ws - 1);
        float acc = 0.0f;
        float out_y = out_y_start;
        for (int64_t in_y = in_y_start; (hb || out_y < fh + 1.0f) && in_y < Hd;) {
            const float yc = __builtin_fmaxf(0.0f, __builtin_fminf(out_y, last_y));
            const float y_lerp = 1.0f - __builtin_fabsf(yc - fh);
            const float yt = __builtin_fminf(__builtin_floorf(yc), last_y);
            const float lepy[2] = {y_lerp, yc - yt};
            float out_x = out_x_start;
            for (int64_t in_x = in_x_start; (wb || out_x < fw + 1.0f) && in_x < Wd;) {
                const int64_t gi = NHWC ? ((n * Hd + in_y) * Wd + in_x) * C + c : ((n * C + c) * Hd + in_y) * Wd + in_x;
                const float gv = ElemIO<TI>::load(g + gi);
                const float xc = __builtin_fmaxf(0.0f, __builtin_fminf(out_x, last_x));
                const float x_lerp = 1.0f - __builtin_fabsf(xc - fw);
                const float xt = __builtin_fminf(__builtin_floorf(xc), last_x);
                const float lepx[2] = {x_lerp, xc - xt};
                if (!hb && !wb) {
                    acc += gv * y_lerp * x_lerp;
                } else if (!hb) {
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        if (xt + (float)j == fw) {
                            acc += gv * lepx[j] * y_lerp;
                        }
                    }
                } else if (!wb) {
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        if (yt + (float)i == fh) {
                            acc += gv * lepy[i] * x_lerp;
                        }
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < 2; i++) {
#pragma unroll
                        for (int j = 0; j < 2; j++) {
                            if (yt + (float)i == fh && xt + (float)j == fw) {
                                acc += gv * lepx[j] * lepy[i];
                            }
                        }
                    }
                }
                in_x++;
                out_x = source_index(scale_w, in_x);
            }
            in_y++;
            out_y = source_index(scale_h, in_y);
        }
        ElemIO<TO>::store(y + idx, acc);
    }
}

template <typename TI, typename TO, bool HALF_PIXEL, bool NHWC>
__global__ __launch_bounds__(kGradThreads) void resize_grad_kernel(const TI* __restrict__ g, TO* __restrict__ y,
                                                                    int64_t total, int32_t C, int32_t Hs, int32_t Ws,
                                                                    int32_t Hd, int32_t Wd, float scale_h,
                                                                    float scale_w, float inv_scale_h,
                                                                    float inv_scale_w)
{
    const int64_t stride = (int64_t)gridDim.x * kGradThreads;
    const float offset = HALF_PIXEL ? 0.5f : 0.0f;
    const float last_y = (float)Hs - 1.0f, last_x = (float)Ws - 1.0f;
    for (int64_t idx = (int64_t)blockIdx.x * kGradThreads + threadIdx.x; idx < total; idx += stride) {
        int64_t t = idx;
        int32_t c, W, H;
        if (NHWC) {
            c = (int32_t)(t % C);
            t /= C;
            W = (int32_t)(t % Ws);
            t /= Ws;
            H = (int32_t)(t % Hs);
            t /= Hs;
        } else {
            W = (int32_t)(t % Ws);
            t /= Ws;
            H = (int32_t)(t % Hs);
            t /= Hs;
            c = (int32_t)(t % C);
            t /= C;
        }
        const int64_t n = t;
        const float fy0 = __builtin_ceilf(((float)H - 1.0f + offset) * inv_scale_h - offset);
        const float fx0 = __builtin_ceilf(((float)W - 1.0f + offset) * inv_scale_w - offset);
        const int64_t in_y_start = (fy0 > 0.0f) ? (int64_t)fy0 : 0;
        const int64_t in_x_start = (fx0 > 0.0f) ? (int64_t)fx0 : 0;
        const float out_y_start = ((float)in_y_start + offset) * scale_h - offset;
        const float out_x_start = ((float)in_x_start + offset) * scale_w - offset;
        const float fh = (float)H, fw = (float)W;
        float acc = 0.0f;
        float out_y = out_y_start;
        for (int64_t in_y = in_y_start; out_y < fh + 1.0f && in_y < Hd; in_y++) {
            const float yc = __builtin_fmaxf(0.0f, __builtin_fminf(out_y, last_y));
            const float y_lerp = 1.0f - __builtin_fabsf(yc - fh);
            float out_x = out_x_start;
            for (int64_t in_x = in_x_start; out_x < fw + 1.0f && in_x < Wd; in_x++) {
                const int64_t gi = NHWC ? ((n * Hd + in_y) * Wd + in_x) * C + c : ((n * C + c) * Hd + in_y) * Wd + in_x;
                const float xc = __builtin_fmaxf(0.0f, __builtin_fminf(out_x, last_x));
                const float x_lerp = 1.0f - __builtin_fabsf(xc - fw);
                acc += ElemIO<TI>::load(g + gi) * y_lerp * x_lerp;
                out_x += scale_w;
            }
            out_y += scale_h;
        }
        ElemIO<TO>::store(y + idx, acc);
    }
}


// LDS-tiled variant of resize_grad_kernel for NCHW.  A workgroup owns (plane, tile of kTileRows x 128 elements of
// the outgoing gradient).  The incoming-gradient rows and columns the tile's lanes will visit form one rectangle
// (start of the first lane, largest end over all lanes, found with the very loops the lanes run later); it is
// copied into LDS with independent 4-byte loads -- all in flight together, where the gather variant waits for one
// two-byte load per visit -- and the lanes then run the unchanged visiting loops on LDS.  A rectangle that does not
// fit the LDS capacity is read from global memory instead (same loops, same result).
// The same sum with the column part of the loop taken out: a lane keeps the weights of the (at most KX) columns it
// visits -- computed once, by the same repeated additions -- and a row costs one LDS read, two products and an add
// per column.  Column k of a lane with fewer than k + 1 visits leaves the sum alone.
template <typename TI, int KX, int KMIN, bool IL = false>
__device__ __forceinline__ float visit_sum_fixed(const TI* tile_xy, int32_t pitch, int32_t y0, int32_t in_y_start,
                                                 int32_t nx, const float* xl, float out_y_start, float fh,
                                                 float scale_h, float last_y, int32_t Hd, float neg_zero,
                                                 int32_t ci = 1)
{
    const int32_t step = IL ? ci : 1;  // elements between the columns a lane visits
    float acc = 0.0f;
    float out_y = out_y_start;
    for (int32_t in_y = in_y_start; out_y < fh + 1.0f && in_y < Hd; in_y++) {
        // max(0, min(out_y, last_y)) as one median: out_y is never a NaN
        const float yc = __builtin_amdgcn_fmed3f(out_y, 0.0f, last_y);
        const float y_lerp = 1.0f - __builtin_fabsf(yc - fh);
        const TI* row = tile_xy + (in_y - y0) * pitch;
#pragma unroll
        for (int k = 0; k < KX; k++) {
            // fma(g, w, -0) is g * w bit for bit and lets a 16-bit element be converted by the multiply itself; the
            // read of a column past the lane's last one may fetch anything (it stays inside LDS) and is dropped.
            // Every lane of the workgroup visits at least KMIN columns: those need no test.
            const float t = __builtin_fmaf(ElemIO<TI>::load(row + k * step), y_lerp, neg_zero) * xl[k];
            acc = (k < KMIN || k < nx) ? acc + t : acc;
        }
        out_y += scale_h;
    }
    return acc;
}

// The same sum once more with the row part taken out as well.  The rows an outgoing row H visits, and their weights,
// do not depend on the plane or the column: a workgroup that walks over planes computes them once per H (by the very
// loop above) and keeps count and weights in registers.  H is the same for all lanes of a wavefront, so the count is
// a scalar and the row loop needs no lane masks.  A visited row then costs the LDS reads, one address add and, per
// column, two products and an add.
constexpr int kRowWeights = 6;  // visited rows per outgoing row kept in registers (more: the loops above)

template <int KX, int KMIN, int Q, bool IL = false>
__device__ __forceinline__ float tile_sum_fixed(const float* lane_rows, int32_t pitch, int32_t n_rows, float lerp_pack,
                                                int32_t nx, const float* xl, float neg_zero, int32_t ci = 1)
{
    const int32_t step = IL ? ci : 1;  // elements between the columns a lane visits
    float acc = 0.0f;
#pragma unroll
    for (int j = 0; j < kRowWeights; j++) {
        if (j < n_rows) {  // n_rows is uniform over the wavefront
            // weight of visited row j of this wavefront's outgoing row Q: lane Q * kRowWeights + j of lerp_pack
            const float y_lerp = __builtin_bit_cast(
                float, __builtin_amdgcn_readlane(__builtin_bit_cast(int32_t, lerp_pack), Q * kRowWeights + j));
#pragma unroll
            for (int k = 0; k < KX; k++) {
                // fma(g, w, -0) is g * w bit for bit; the compiler may not fold it into the following product
                const float t = __builtin_fmaf(lane_rows[k * step], y_lerp, neg_zero) * xl[k];
                acc = (k < KMIN || k < nx) ? acc + t : acc;
            }
            lane_rows += pitch;
        }
    }
    return acc;
}

// IL: channels-last tensors, taken as planes whose rows are W * ci elements (element j of a row is channel j % ci of
// pixel j / ci); "columns" then count row elements, a lane's visited columns sit ci elements apart, and the column
// geometry (first visit, count, weights) is that of the lane's pixel.
template <typename TI, typename TO, bool HALF_PIXEL, bool IL>
__global__ __launch_bounds__(kGradThreads) void resize_grad_lds_kernel(const TI* __restrict__ g, TO* __restrict__ y,
                                                                        int64_t planes, int32_t Hs, int32_t Ws,
                                                                        int32_t Hd, int32_t Wd, float scale_h,
                                                                        float scale_w, float inv_scale_h,
                                                                        float inv_scale_w, int32_t tile_rows,
                                                                        int32_t cap_words, float neg_zero,
                                                                        uint32_t tiles_x, uint32_t tiles_y,
                                                                        uint32_t plane_slots, int32_t ci_arg)
{
    const int32_t ci = IL ? ci_arg : 1;
    const int32_t Wse = Ws * ci, Wde = Wd * ci;  // row elements
    // Workgroups are handed to the eight XCDs in turn, each with its own L2.  The launch is one-dimensional and padded
    // to a multiple of eight; workgroup L becomes tile (L % 8) * (count / 8) + L / 8, so that an XCD works through a
    // contiguous run of tiles and the rows and 128-byte lines that neighbouring tiles share are fetched from memory
    // once per XCD rather than once per tile.
    const uint32_t per_xcd = gridDim.x / 8u;
    const uint32_t tile_id = (blockIdx.x % 8u) * per_xcd + blockIdx.x / 8u;
    if (tile_id >= tiles_x * tiles_y * plane_slots) {
        return;
    }
    const uint32_t block_x = tile_id % tiles_x, block_y = (tile_id / tiles_x) % tiles_y;
    const uint32_t block_z = tile_id / (tiles_x * tiles_y);
    constexpr int EPW = 4 / (int)sizeof(TI);  // elements per 4-byte word
    extern __shared__ __attribute__((aligned(16))) uint32_t tile_words[];
    __shared__ int32_t s_x1, s_y1, s_nx, s_nx_min;
    const int tx = threadIdx.x % kGradTileCols, ty = threadIdx.x / kGradTileCols;
    const int32_t W0 = (int32_t)block_x * kGradTileCols, H0 = (int32_t)block_y * tile_rows;
    const float offset = HALF_PIXEL ? 0.5f : 0.0f;
    const float last_y = (float)Hs - 1.0f, last_x = (float)Ws - 1.0f;
    auto first_visit = [&](int32_t i, float inv_scale, int32_t len_dst) {
        const float f = __builtin_ceilf(((float)i - 1.0f + offset) * inv_scale - offset);
        // a start at or beyond the end visits nothing, whatever its exact value
        return (f > 0.0f) ? ((f < (float)len_dst) ? (int32_t)f : len_dst) : 0;
    };
    auto end_visit = [&](int32_t i, int32_t start, float scale, int32_t len_dst) {
        float out = ((float)start + offset) * scale - offset;
        int32_t in = start;
        for (; out < (float)i + 1.0f && in < len_dst; in++) {
            out += scale;
        }
        return in;
    };
    const int32_t W = W0 + tx;
    const bool col_ok = W < Wse;
    const int32_t px = IL ? (col_ok ? W : W0) / ci : (col_ok ? W : W0);  // pixel of this lane's column
    const int32_t ch = IL ? (col_ok ? W : W0) - px * ci : 0;               // and its channel
    const int32_t in_x_start = first_visit(px, inv_scale_w, Wd);
    const int32_t tile_x0 = first_visit(IL ? W0 / ci : W0, inv_scale_w, Wd) * ci / EPW * EPW;
    const int32_t tile_y0 = first_visit(H0, inv_scale_h, Hd);
    if (threadIdx.x == 0) {
        s_x1 = 0;
        s_y1 = 0;
        s_nx = 0;
        s_nx_min = INT32_MAX;
    }
    __syncthreads();
    int32_t nx = 0;
    {
        // largest end and largest visit count over the wavefront by a butterfly of lane exchanges, then one LDS atomic
        // per wavefront (an atomic per lane is serialised lane by lane on the scalar unit)
        int32_t x_end = 0;
        if (col_ok) {
            x_end = end_visit(px, in_x_start, scale_w, Wd);
            nx = x_end - in_x_start;
        }
        int32_t m_end = x_end, m_nx = nx, m_min = col_ok ? nx : INT32_MAX;  // lanes past the last column do not count
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) {
            const int32_t o_end = __shfl_xor(m_end, d), o_nx = __shfl_xor(m_nx, d), o_min = __shfl_xor(m_min, d);
            m_end = (o_end > m_end) ? o_end : m_end;
            m_nx = (o_nx > m_nx) ? o_nx : m_nx;
            m_min = (o_min < m_min) ? o_min : m_min;
        }
        if ((threadIdx.x & 63) == 0) {
            atomicMax(&s_x1, m_end);
            atomicMax(&s_nx, m_nx);
            atomicMin(&s_nx_min, m_min);
        }
    }
    if (tx == 0) {
        for (int32_t H = H0 + ty; H < H0 + tile_rows && H < Hs; H += kGradTileGroups) {
            atomicMax(&s_y1, end_visit(H, first_visit(H, inv_scale_h, Hd), scale_h, Hd));
        }
    }
    __syncthreads();
    const int32_t tile_x1 = (s_x1 * ci + EPW - 1) / EPW * EPW;  // rows are multiples of EPW (host check): stays inside
    const int32_t tile_y1 = s_y1;
    const int32_t pitch_w = (tile_x1 > tile_x0) ? (tile_x1 - tile_x0) / EPW : 0;
    const int32_t rows = (tile_y1 > tile_y0) ? tile_y1 - tile_y0 : 0;
    // the tile holds fp32 values (16-bit gradients are widened by the copy, which is exact): a lane's run of columns
    // then starts on a 4-byte boundary whatever its parity, and LDS reads that straddle words are several times slower
    const int32_t pitch = pitch_w * EPW;
    const bool use_lds = (int64_t)rows * pitch <= cap_words;
    const float* tile = reinterpret_cast<const float*>(tile_words);
    const float out_x_start = ((float)in_x_start + offset) * scale_w - offset;
    const float fw = (float)px;

    // column weights of this lane, for the variants with a fixed column count
    constexpr int KMAX = 8;
    float xl[KMAX];
    {
        float out_x = out_x_start;
#pragma unroll
        for (int k = 0; k < KMAX; k++) {
            const float xc = __builtin_fmaxf(0.0f, __builtin_fminf(out_x, last_x));
            xl[k] = 1.0f - __builtin_fabsf(xc - fw);
            out_x += scale_w;
        }
    }
    const int32_t nx_max = s_nx, nx_min = s_nx_min;
    // starting position and step of this lane in the tile's (row, word) grid for the copy loop
    const int32_t pw1 = (pitch_w > 0) ? pitch_w : 1;
    const int32_t ld_r0 = (int32_t)threadIdx.x / pw1, ld_c0 = (int32_t)threadIdx.x % pw1;
    const int32_t ld_dr = kGradThreads / pw1, ld_dc = kGradThreads % pw1;
    const int32_t x_base = (nx > 0) ? in_x_start * ci + ch - tile_x0 : 0;

    // rows visited by each of this wavefront's outgoing rows, and their weights (see tile_sum_fixed)
    constexpr int HQ = 8 / kGradTileGroups;  // outgoing rows per lane at the largest tile height
    static_assert(HQ * kRowWeights <= 64, "the row weights of a wavefront are packed one per lane");
    float lerp_pack = 0.0f;  // lane q * kRowWeights + j: weight of visited row j of outgoing row q (a uniform table)
    int32_t meta_pack = -1;  // lane q: rows outgoing row q visits (-1: no such row in this tile); lane 8 + q: the first
    bool rows_fixed = true;
    const int32_t lane_id = (int32_t)threadIdx.x & 63;
#pragma unroll
    for (int q = 0; q < HQ; q++) {
        const int32_t H = __builtin_amdgcn_readfirstlane(H0 + ty + q * kGradTileGroups);
        if (H < H0 + tile_rows && H < Hs) {
            const int32_t start = first_visit(H, inv_scale_h, Hd);
            float out_y = ((float)start + offset) * scale_h - offset;
            const float fh = (float)H;
            int32_t n = 0;
            for (int32_t in_y = start; out_y < fh + 1.0f && in_y < Hd; in_y++) {
                const float w = 1.0f - __builtin_fabsf(__builtin_amdgcn_fmed3f(out_y, 0.0f, last_y) - fh);
                lerp_pack = (n < kRowWeights && lane_id == q * kRowWeights + n) ? w : lerp_pack;
                n++;
                out_y += scale_h;
            }
            meta_pack = (lane_id == q) ? n : ((lane_id == 8 + q) ? start : meta_pack);
            rows_fixed = rows_fixed && (__builtin_amdgcn_readfirstlane(n) <= kRowWeights);
        }
    }

    // Copy of the rectangle into LDS: word i of the tile is (row i / pitch_w, word i % pitch_w) of the rectangle.
    const int32_t total = rows * pitch_w;
    const int32_t row_words = Wde / EPW;

    for (int64_t pl = block_z; pl < planes; pl += plane_slots) {
        const TI* gp = g + pl * (int64_t)Hd * Wde;
        if (use_lds) {
            // the pair (row, word) is advanced instead of divided
            int32_t r = ld_r0, cw = ld_c0;
            const uint32_t* src = reinterpret_cast<const uint32_t*>(gp + (int64_t)tile_y0 * Wde + tile_x0);
#pragma unroll 8
            for (int32_t i = threadIdx.x; i < total; i += kGradThreads) {
                const uint32_t word = src[(int64_t)r * row_words + cw];
                if (EPW == 1) {
                    tile_words[i] = word;
                } else {
                    TI pair[2];
                    __builtin_memcpy(pair, &word, 4);
                    float2 wide;
                    wide.x = ElemIO<TI>::load(&pair[0]);
                    wide.y = ElemIO<TI>::load(&pair[1]);
                    reinterpret_cast<float2*>(tile_words)[i] = wide;
                }
                r += ld_dr;
                cw += ld_dc;
                if (cw >= pitch_w) {
                    cw -= pitch_w;
                    r++;
                }
            }
            __syncthreads();
        }
        if (col_ok && use_lds && rows_fixed && nx_max <= 6) {
            TO* yp = y + (pl * Hs + H0 + ty) * (int64_t)Wse + W;
            // -0 in a vector register: with the row weight in a scalar one, a second scalar operand would be copied
            // into a vector register before every product
            const float neg_zero_v = as_fp32_value(neg_zero);
            auto one_row = [&](auto qc) {
                constexpr int q = decltype(qc)::value;
                // read where they are used: kept in scalar registers from the set-up on, they would be spilled
                const int32_t n_rows = __builtin_amdgcn_readlane(meta_pack, q);
                if (n_rows >= 0) {
                    const int32_t first_row = __builtin_amdgcn_readlane(meta_pack, 8 + q);
                    const float* lane_rows = tile + (first_row - tile_y0) * pitch + x_base;
                    float acc;
#define OPSCV_TILE_SUM(KX, KMIN) \
    tile_sum_fixed<KX, KMIN, q, IL>(lane_rows, pitch, n_rows, lerp_pack, nx, xl, neg_zero_v, ci)
                    if (nx_max <= 4) {
                        acc = (nx_min >= 4) ? OPSCV_TILE_SUM(4, 4) : OPSCV_TILE_SUM(4, 0);
                    } else if (nx_max <= 5) {
                        acc = (nx_min >= 4) ? OPSCV_TILE_SUM(5, 4) : OPSCV_TILE_SUM(5, 0);
                    } else {
                        acc = (nx_min >= 4) ? OPSCV_TILE_SUM(6, 4) : OPSCV_TILE_SUM(6, 0);
                    }
#undef OPSCV_TILE_SUM
                    store_streaming<TO>(yp + (int64_t)q * kGradTileGroups * Wse, acc);
                }
            };
            static_assert(HQ == 4, "one call per outgoing row of a lane");
            one_row(std::integral_constant<int, 0>{});
            one_row(std::integral_constant<int, 1>{});
            one_row(std::integral_constant<int, 2>{});
            one_row(std::integral_constant<int, 3>{});
        } else if (col_ok) {
            for (int32_t H = H0 + ty; H < H0 + tile_rows && H < Hs; H += kGradTileGroups) {
                const int32_t in_y_start = first_visit(H, inv_scale_h, Hd);
                const float out_y_start = ((float)in_y_start + offset) * scale_h - offset;
                float acc;
                // separate call sites so that each is compiled for its own address space (LDS reads, global loads)
#define OPSCV_VISIT(KX, KMIN)                                                                                       \
    visit_sum_fixed<float, KX, KMIN, IL>(tile + x_base, pitch, tile_y0, in_y_start, nx, xl, out_y_start, (float)H,    \
                                         scale_h, last_y, Hd, neg_zero, ci)
                if (use_lds && nx_max <= 4) {
                    acc = (nx_min >= 4) ? OPSCV_VISIT(4, 4) : OPSCV_VISIT(4, 0);
                } else if (use_lds && nx_max <= 5) {
                    acc = (nx_min >= 4) ? OPSCV_VISIT(5, 4) : OPSCV_VISIT(5, 0);
                } else if (use_lds && nx_max <= 6) {
                    acc = (nx_min >= 4) ? OPSCV_VISIT(6, 4) : OPSCV_VISIT(6, 0);
                } else if (use_lds && nx_max <= 8) {
                    acc = OPSCV_VISIT(8, 0);
                } else if (use_lds) {
                    acc = visit_sum<float>(tile, pitch, tile_y0, tile_x0, in_y_start, in_x_start, out_y_start,
                                        out_x_start, (float)H, fw, scale_h, scale_w, last_y, last_x, Hd, Wd, ci, ch);
                } else {
                    acc = visit_sum<TI>(gp, Wde, 0, 0, in_y_start, in_x_start, out_y_start, out_x_start, (float)H, fw,
                                        scale_h, scale_w, last_y, last_x, Hd, Wd, ci, ch);
                }
#undef OPSCV_VISIT
                store_streaming<TO>(y + (pl * Hs + H) * (int64_t)Wse + W, acc);
            }
        }
        if (use_lds) {
            __syncthreads();  // the tile is overwritten by the next plane
        }
    }
}

// Planes whose elements grow by up to four a side (at most eight visited rows and columns) and that resize_grad_rows.hip leaves
// (rows_plan: mostly fp32 planes of 42 to 63 columns, and of up to three columns): the rectangle stays in the element type and
// comes by asynchronous copies.
//
// A workgroup owns 64 outgoing columns by 16 or 8 outgoing rows, a wavefront every fourth of the rows.  The row segments
// the tile visits are copied from the 16-byte boundary before their first byte to the one after their last (the bytes
// outside share an aligned unit with bytes inside, so they are readable), so rows may have any length and start at any
// element; where a row then starts in LDS is uniform, and a lane reads its run of columns from the 4-byte word its first
// one lies in.  16-bit columns are shifted into place pair by pair: the reads never straddle a word, and a run takes
// half the LDS traffic of fp32 words, whose lanes meet in one bank in four where the columns grow by four.
// Same visits, products and order of the sum as resize_grad_kernel.
//
// What bounds it: vector instructions, three per visit plus the shifts, and the set-up of a tile where it serves few
// planes.  bf16 8x64x65x129 from 257x513: 55 us, 72 before the one column past whole tiles was taken by strip_element, and 189
// in resize_grad_kernel, where rows of odd length were left before.  4x32x160x240 against resize_grad_lds_kernel (fp16 even rows / fp32) and the gather (bf16 odd rows), before ->
// after: growth by 0.6 24 -> 16 / 24 -> 16 / 28 -> 17 us, by two 38 -> 29 / 40 -> 28 / 63 -> 31, by three 95 -> 51 /
// 105 -> 47 / 118 -> 45, by four 136 -> 57 / 174 -> 109 (a growth above four: the gather as before).
typedef __attribute__((address_space(1))) const void* rg_global_cptr_t;
typedef __attribute__((address_space(3))) void* rg_lds_ptr_t;

// Columns 0 .. KX - 1 of the run that starts at LDS byte `off`, times y_lerp (fma(g, w, -0) is g * w bit for bit).
template <typename TI, int KX>
__device__ __forceinline__ void weighted_columns(const char* lds, uint32_t off, float y_lerp, float neg_zero, float* t)
{
    if constexpr (sizeof(TI) == 4) {
        const float* w = reinterpret_cast<const float*>(lds + off);
#pragma unroll
        for (int k = 0; k < KX; k++) {
            t[k] = w[k] * y_lerp;
        }
    } else {
        constexpr int PAIRS = (KX + 1) / 2;
        const uint32_t* w = reinterpret_cast<const uint32_t*>(lds + (off & ~3u));
        const uint32_t bits = off << 3;  // alignbit takes its low five bits: 0 or 16
        uint32_t word[PAIRS + 1];
#pragma unroll
        for (int k = 0; k <= PAIRS; k++) {
            word[k] = w[k];
        }
#pragma unroll
        for (int k = 0; k < PAIRS; k++) {
            const uint32_t both = __builtin_amdgcn_alignbit(word[k + 1], word[k], bits);
            TI pair[2];
            __builtin_memcpy(pair, &both, 4);
            t[2 * k] = __builtin_fmaf(ElemIO<TI>::load(&pair[0]), y_lerp, neg_zero);
            if (2 * k + 1 < KX) {
                t[2 * k + 1] = __builtin_fmaf(ElemIO<TI>::load(&pair[1]), y_lerp, neg_zero);
            }
        }
    }
}

// Element e of the columns past the last whole tile, all planes' one after the other: a lane each, straight from memory, the
// up to eight loads of a row on their way together.  These workgroups go first, so that their chain of a load a row ends
// under the tiles'.
template <typename TI, typename TO, bool HALF_PIXEL>
__device__ __forceinline__ void strip_element(const TI* __restrict__ g, TO* __restrict__ y, int64_t planes, int32_t Hs,
                                              int32_t Ws, int32_t Hd, int32_t Wd, float scale_h, float scale_w,
                                              float inv_scale_h, float inv_scale_w, uint32_t cols, uint32_t e)
{
    const uint32_t line = e / cols, pl = line / (uint32_t)Hs;
    if ((int64_t)pl >= planes) {
        return;
    }
    const int32_t H = (int32_t)(line - pl * (uint32_t)Hs), W = Ws - (int32_t)cols + (int32_t)(e - line * cols);
    const float offset = HALF_PIXEL ? 0.5f : 0.0f, fh = (float)H, fw = (float)W;
    const float last_y = (float)Hs - 1.0f, last_x = (float)Ws - 1.0f;
    const int32_t in_x_start = first_visited<HALF_PIXEL>(W, inv_scale_w, Wd);
    const int32_t in_y_start = first_visited<HALF_PIXEL>(H, inv_scale_h, Hd);
    const float out_x_start = ((float)in_x_start + offset) * scale_w - offset;
    const float out_y_start = ((float)in_y_start + offset) * scale_h - offset;
    const TI* gp = g + (int64_t)pl * Hd * Wd;
    int32_t nx = 0;
    float xl[kPlaneVisits], out_x = out_x_start;
#pragma unroll
    for (int k = 0; k < kPlaneVisits; k++) {
        xl[k] = 1.0f - __builtin_fabsf(__builtin_fmaxf(0.0f, __builtin_fminf(out_x, last_x)) - fw);
        out_x += scale_w;
    }
    out_x = out_x_start;
    for (int32_t in_x = in_x_start; out_x < fw + 1.0f && in_x < Wd; in_x++) {
        nx++;
        out_x += scale_w;
    }
    float acc = 0.0f;
    if (nx > kPlaneVisits) {
        acc = visit_sum<TI>(gp, Wd, 0, 0, in_y_start, in_x_start, out_y_start, out_x_start, fh, fw, scale_h, scale_w, last_y,
                            last_x, Hd, Wd);
    } else if (nx > 0) {
        float out_y = out_y_start;
#pragma unroll 2
        for (int32_t in_y = in_y_start; out_y < fh + 1.0f && in_y < Hd; in_y++) {
            const float y_lerp = 1.0f - __builtin_fabsf(__builtin_fmaxf(0.0f, __builtin_fminf(out_y, last_y)) - fh);
            const TI* row = gp + (int64_t)in_y * Wd + in_x_start;
            TI v[kPlaneVisits];
#pragma unroll
            for (int k = 0; k < kPlaneVisits; k++) {
                v[k] = row[k < nx ? k : 0];
            }
#pragma unroll
            for (int k = 0; k < kPlaneVisits; k++) {
                const float t = ElemIO<TI>::load(&v[k]) * y_lerp * xl[k];
                acc = (k < nx) ? acc + t : acc;
            }
            out_y += scale_h;
        }
    }
    store_streaming<TO>(y + (int64_t)pl * Hs * Ws + (int64_t)H * Ws + W, acc);
}

template <typename TI, typename TO, bool HALF_PIXEL>
__global__ __launch_bounds__(kGradThreads) void resize_grad_planes_kernel(
    const TI* __restrict__ g, TO* __restrict__ y, int64_t planes, int32_t Hs, int32_t Ws, int32_t Hd, int32_t Wd,
    float scale_h, float scale_w, float inv_scale_h, float inv_scale_w, int32_t tile_rows, int32_t lds_bytes,
    float neg_zero, uint32_t tiles_x, uint32_t tiles_y, uint32_t plane_slots, uint32_t strip_cols, uint32_t strip_blocks)
{
    if (blockIdx.x < strip_blocks) {
        strip_element<TI, TO, HALF_PIXEL>(g, y, planes, Hs, Ws, Hd, Wd, scale_h, scale_w, inv_scale_h, inv_scale_w, strip_cols,
                                          blockIdx.x * kGradThreads + threadIdx.x);
        return;
    }
    // tiles go to the XCDs as in resize_grad_lds_kernel; the strip's workgroups are whole eights
    const uint32_t tile_block = blockIdx.x - strip_blocks, per_xcd = (gridDim.x - strip_blocks) / 8u;
    const uint32_t tile_id = (tile_block % 8u) * per_xcd + tile_block / 8u;
    if (tile_id >= tiles_x * tiles_y * plane_slots) {
        return;
    }
    const uint32_t block_x = tile_id % tiles_x, block_y = (tile_id / tiles_x) % tiles_y;
    const uint32_t block_z = tile_id / (tiles_x * tiles_y);
    constexpr int NWAVES = kGradThreads / 64;
    constexpr int HQ = kPlaneRows / NWAVES;  // outgoing rows of a wavefront at the largest tile height
    static_assert(HQ * kPlaneVisits <= 64, "the row weights of a wavefront are packed one per lane");
    extern __shared__ __attribute__((aligned(16))) uint32_t tile_words[];
    __shared__ int32_t s_x1, s_y1, s_nx, s_nx_min;
    char* lds = reinterpret_cast<char*>(tile_words);
    const int32_t lane = (int32_t)threadIdx.x & 63;
    const int32_t wave = __builtin_amdgcn_readfirstlane((int32_t)threadIdx.x >> 6);
    const int32_t W0 = (int32_t)block_x * kPlaneCols, H0 = (int32_t)block_y * tile_rows;
    const float offset = HALF_PIXEL ? 0.5f : 0.0f;
    const float last_y = (float)Hs - 1.0f, last_x = (float)Ws - 1.0f;
    auto first_visit = [&](int32_t i, float inv_scale, int32_t len_dst) {
        return first_visited<HALF_PIXEL>(i, inv_scale, len_dst);
    };
    const int32_t W = W0 + lane;
    const bool col_ok = W < Ws;
    const int32_t col = col_ok ? W : W0;
    const float fw = (float)col;
    const int32_t in_x_start = first_visit(col, inv_scale_w, Wd);
    const int32_t tile_x0 = first_visit(W0, inv_scale_w, Wd);
    const int32_t tile_y0 = first_visit(H0, inv_scale_h, Hd);
    const float out_x_start = ((float)in_x_start + offset) * scale_w - offset;
    if (threadIdx.x == 0) {
        s_y1 = 0;
    }
    __syncthreads();

    // The columns this lane visits and their weights, by the loop of resize_grad_kernel; the rows each of the wavefront's
    // outgoing rows visits and theirs, one per lane (the row is the same for all lanes).
    int32_t nx = 0;
    float xl[kPlaneVisits];
    {
        float out_x = out_x_start;
#pragma unroll
        for (int k = 0; k < kPlaneVisits; k++) {
            xl[k] = 1.0f - __builtin_fabsf(__builtin_fmaxf(0.0f, __builtin_fminf(out_x, last_x)) - fw);
            out_x += scale_w;
        }
        out_x = out_x_start;
        for (int32_t in_x = in_x_start; out_x < fw + 1.0f && in_x < Wd; in_x++) {
            nx++;
            out_x += scale_w;
        }
    }
    float lerp_pack = 0.0f;  // lane q * kPlaneVisits + j: weight of visited row j of outgoing row q
    int32_t meta_pack = -1;  // lane q: rows outgoing row q visits (-1: no such row in this tile); lane 8 + q: the first
    bool fits = true;
    int32_t y_end = 0;
    static_assert(HQ <= 8, "counts in lanes 0 to 7, first rows in lanes 8 to 15");
    for (int q = 0; q < HQ; q++) {
        const int32_t H = H0 + wave + q * NWAVES;
        if (H < H0 + tile_rows && H < Hs) {
            const int32_t start = first_visit(H, inv_scale_h, Hd);
            float out_y = ((float)start + offset) * scale_h - offset;
            const float fh = (float)H;
            int32_t n = 0;
            for (int32_t in_y = start; out_y < fh + 1.0f && in_y < Hd; in_y++) {
                const float w = 1.0f - __builtin_fabsf(__builtin_amdgcn_fmed3f(out_y, 0.0f, last_y) - fh);
                lerp_pack = (n < kPlaneVisits && lane == q * kPlaneVisits + n) ? w : lerp_pack;
                n++;
                out_y += scale_h;
            }
            n = __builtin_amdgcn_readfirstlane(n);
            meta_pack = (lane == q) ? n : ((lane == 8 + q) ? start : meta_pack);
            fits = fits && n <= kPlaneVisits;
            y_end = (start + n > y_end) ? start + n : y_end;
        }
    }
    {
        // largest end and visit counts over the wavefront's columns, which are the workgroup's
        int32_t m_end = col_ok ? in_x_start + nx : 0, m_nx = col_ok ? nx : 0, m_min = col_ok ? nx : INT32_MAX;
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) {
            const int32_t o_end = __shfl_xor(m_end, d), o_nx = __shfl_xor(m_nx, d), o_min = __shfl_xor(m_min, d);
            m_end = (o_end > m_end) ? o_end : m_end;
            m_nx = (o_nx > m_nx) ? o_nx : m_nx;
            m_min = (o_min < m_min) ? o_min : m_min;
        }
        if (threadIdx.x == 0) {
            s_x1 = m_end;
            s_nx = m_nx;
            s_nx_min = m_min;
        }
        if (lane == 0) {
            atomicMax(&s_y1, fits ? y_end : INT32_MAX);  // a row of too many visits: no rectangle is large enough
        }
    }
    __syncthreads();
    const int32_t tile_x1 = __builtin_amdgcn_readfirstlane(s_x1), tile_y1 = __builtin_amdgcn_readfirstlane(s_y1);
    const int32_t nx_max = __builtin_amdgcn_readfirstlane(s_nx), nx_min = __builtin_amdgcn_readfirstlane(s_nx_min);
    const int32_t rows = (tile_y1 > tile_y0) ? tile_y1 - tile_y0 : 0;
    const uint32_t seg_bytes = (tile_x1 > tile_x0) ? (uint32_t)(tile_x1 - tile_x0) * (uint32_t)sizeof(TI) : 0u;
    const uint32_t pitch = (seg_bytes + 30u) & ~15u;
    const bool use_lds = nx_max <= kPlaneVisits && (int64_t)rows * pitch + kPlanePad <= lds_bytes;
    const uint32_t lane_off = (nx > 0) ? (uint32_t)(in_x_start - tile_x0) * (uint32_t)sizeof(TI) : 0u;
    const uint32_t row_low = ((uint32_t)Wd * (uint32_t)sizeof(TI)) & 15u;
    const float neg_zero_v = as_fp32_value(neg_zero);

    for (int64_t pl = block_z; pl < planes; pl += plane_slots) {
        const TI* gp = g + pl * (int64_t)Hd * Wd;
        TO* yp = y + pl * (int64_t)Hs * Ws + W;
        if (!use_lds) {
            for (int32_t H = H0 + wave; col_ok && H < H0 + tile_rows && H < Hs; H += NWAVES) {
                const int32_t in_y_start = first_visit(H, inv_scale_h, Hd);
                const float out_y_start = ((float)in_y_start + offset) * scale_h - offset;
                store_streaming<TO>(yp + (int64_t)H * Ws,
                                    visit_sum<TI>(gp, Wd, 0, 0, in_y_start, in_x_start, out_y_start, out_x_start, (float)H,
                                                  fw, scale_h, scale_w, last_y, last_x, Hd, Wd));
            }
            continue;
        }
        const char* src0 = reinterpret_cast<const char*>(gp + (int64_t)tile_y0 * Wd + tile_x0);
        const uint32_t src0_low = (uint32_t)(reinterpret_cast<uintptr_t>(src0) & 15u);
        // bytes by which the copy of staged row r starts before the row's segment
        auto row_shift = [&](uint32_t r) -> uint32_t { return (src0_low + r * row_low) & 15u; };
        for (uint32_t r = (uint32_t)wave; r < (uint32_t)rows; r += NWAVES) {
            const uint32_t shift = row_shift(r);
            const uint32_t limit = (seg_bytes + shift + 15u) & ~15u;
            const char* row = src0 + (int64_t)r * Wd * (int64_t)sizeof(TI) - shift;
            for (uint32_t cb = 0; cb < limit; cb += 1024u) {
                const uint32_t at = cb + (uint32_t)lane * 16u;
                if (at < limit) {
                    __builtin_amdgcn_global_load_lds((rg_global_cptr_t)(row + at), (rg_lds_ptr_t)(lds + r * pitch + cb), 16,
                                                     0, 0);
                }
            }
        }
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        // KX: columns read, at least as many as any lane visits; every lane visits at least KMIN
        auto sums = [&](auto kx, auto kmin) {
            constexpr int KX = decltype(kx)::value, KMIN = decltype(kmin)::value;
            for (int q = 0; q < HQ; q++) {
                const int32_t n_rows = __builtin_amdgcn_readlane(meta_pack, q);
                if (n_rows < 0) {
                    break;
                }
                uint32_t r = (uint32_t)(__builtin_amdgcn_readlane(meta_pack, 8 + q) - tile_y0);
                float acc = 0.0f;
#pragma unroll 2
                for (int j = 0; j < n_rows; j++, r++) {
                    const float y_lerp = __builtin_bit_cast(
                        float, __builtin_amdgcn_readlane(__builtin_bit_cast(int32_t, lerp_pack), q * kPlaneVisits + j));
                    float t[KX + 1];
                    weighted_columns<TI, KX>(lds, lane_off + (r * pitch + row_shift(r)), y_lerp, neg_zero_v, t);
#pragma unroll
                    for (int k = 0; k < KX; k++) {
                        const float v = t[k] * xl[k];
                        acc = (k < KMIN || k < nx) ? acc + v : acc;
                    }
                }
                if (col_ok) {
                    store_streaming<TO>(yp + (int64_t)(H0 + wave + q * NWAVES) * Ws, acc);
                }
            }
        };
        typedef std::integral_constant<int, 0> k0;
        typedef std::integral_constant<int, 4> k4;
        if (nx_max <= 2) {
            sums(std::integral_constant<int, 2>{}, k0{});
        } else if (nx_max <= 4) {
            (nx_min >= 4) ? sums(k4{}, k4{}) : sums(k4{}, k0{});
        } else if (nx_max <= 5) {
            (nx_min >= 4) ? sums(std::integral_constant<int, 5>{}, k4{}) : sums(std::integral_constant<int, 5>{}, k0{});
        } else if (nx_max <= 6) {
            (nx_min >= 4) ? sums(std::integral_constant<int, 6>{}, k4{}) : sums(std::integral_constant<int, 6>{}, k0{});
        } else {
            (nx_min >= 6) ? sums(std::integral_constant<int, 8>{}, std::integral_constant<int, 6>{})
                          : sums(std::integral_constant<int, 8>{}, k0{});
        }
        __syncthreads();  // the tile is overwritten by the next plane
    }
}

template <typename TI, typename TO>
hipError_t run_planes(const ResizeGradArgs& a, const PlaneTile& t, hipStream_t stream)
{
    const int64_t planes = a.N * a.C;
#define OPSCV_RGP(HP)                                                                                                \
    hipLaunchKernelGGL((resize_grad_planes_kernel<TI, TO, HP>), dim3((unsigned)t.blocks), dim3(kGradThreads),        \
                       t.lds_bytes, stream, (const TI*)a.x, (TO*)a.y, planes, (int32_t)a.Hs, (int32_t)a.Ws,          \
                       (int32_t)a.Hd, (int32_t)a.Wd, a.scale_h, a.scale_w, a.inv_scale_h, a.inv_scale_w, t.rows,     \
                       t.lds_bytes, -0.0f, (uint32_t)t.tiles_x, (uint32_t)t.tiles_y, (uint32_t)t.slots,       \
                       (uint32_t)t.strip_cols, (uint32_t)t.strip_blocks)
    if (a.half_pixel) {
        OPSCV_RGP(true);
    } else {
        OPSCV_RGP(false);
    }
#undef OPSCV_RGP
    return hipGetLastError();
}

template <typename TI, typename TO>
hipError_t run(const ResizeGradArgs& a, hipStream_t stream)
{
    const ResizeGradPlan plan = resize_grad_plan(a);
    if (plan.kernel == ResizeGradKernel::Rows) {
        return run_resize_grad_rows(a, plan.rows, stream);
    }
    if (plan.kernel == ResizeGradKernel::Planes) {
        return run_planes<TI, TO>(a, plan.planes, stream);
    }
    if (plan.kernel == ResizeGradKernel::Lds) {
        const LdsTile& t = plan.lds;
        const int32_t ci = (int32_t)(a.channels_last ? a.C : 1);
        const int64_t planes = a.channels_last ? a.N : a.N * a.C;
#define OPSCV_RGL(HP, IL)                                                                                            \
    hipLaunchKernelGGL((resize_grad_lds_kernel<TI, TO, HP, IL>), dim3((unsigned)t.blocks), dim3(kGradThreads),           \
                       t.lds_words * 4, stream,                                                                      \
                       (const TI*)a.x, (TO*)a.y, planes, (int32_t)a.Hs, (int32_t)a.Ws, (int32_t)a.Hd, (int32_t)a.Wd, \
                       a.scale_h, a.scale_w, a.inv_scale_h, a.inv_scale_w, t.rows, t.lds_words, -0.0f,               \
                       (uint32_t)t.tiles_x, (uint32_t)t.tiles_y, (uint32_t)t.slots, ci)
        if (a.half_pixel) {
            if (a.channels_last) {
                OPSCV_RGL(true, true);
            } else {
                OPSCV_RGL(true, false);
            }
        } else {
            if (a.channels_last) {
                OPSCV_RGL(false, true);
            } else {
                OPSCV_RGL(false, false);
            }
        }
#undef OPSCV_RGL
        return hipGetLastError();
    }
    const int64_t total = a.N * a.C * a.Hs * a.Ws;
    int64_t blocks = (total + kGradThreads - 1) / kGradThreads;
    if (blocks > 256 * 256) {
        blocks = 256 * 256;
    }
#define OPSCV_RG(HP, CL)                                                                                              \
    if (a.user_scales) {                                                                                              \
        hipLaunchKernelGGL((resize_grad_scales_kernel<TI, TO, HP, CL>), dim3((unsigned)blocks), dim3(kGradThreads),   \
                           0, stream, (const TI*)a.x, (TO*)a.y, total, (int32_t)a.C, (int32_t)a.Hs, (int32_t)a.Ws,    \
                           (int32_t)a.Hd, (int32_t)a.Wd, a.scale_h, a.scale_w, a.inv_scale_h, a.inv_scale_w);         \
    } else {                                                                                                          \
        hipLaunchKernelGGL((resize_grad_kernel<TI, TO, HP, CL>), dim3((unsigned)blocks), dim3(kGradThreads), 0,       \
                           stream, (const TI*)a.x, (TO*)a.y, total, (int32_t)a.C, (int32_t)a.Hs, (int32_t)a.Ws,       \
                           (int32_t)a.Hd, (int32_t)a.Wd, a.scale_h, a.scale_w, a.inv_scale_h, a.inv_scale_w);         \
    }
    if (a.half_pixel) {
        if (a.channels_last) {
            OPSCV_RG(true, true);
        } else {
            OPSCV_RG(true, false);
        }
    } else {
        if (a.channels_last) {
            OPSCV_RG(false, true);
        } else {
            OPSCV_RG(false, false);
        }
    }
#undef OPSCV_RG
    return hipGetLastError();
}

}  // namespace

const char* resize_grad_variant(const ResizeGradArgs& a)
{
    switch (resize_grad_plan(a).kernel) {
        case ResizeGradKernel::Scales: return "resize_grad_gather_scales";
        case ResizeGradKernel::Rows: return "resize_grad_rows";
        case ResizeGradKernel::Planes:
        case ResizeGradKernel::Lds: return "resize_grad_lds";
        case ResizeGradKernel::Gather: break;
    }
    return "resize_grad_gather";
}

hipError_t launch_resize_grad(const ResizeGradArgs& a, hipStream_t stream)
{
    const int64_t lim = INT32_MAX;
    if (a.N < 0 || a.C < 0 || a.Hs <= 0 || a.Ws <= 0 || a.Hd <= 0 || a.Wd <= 0 || a.Hs > lim || a.Ws > lim ||
        a.Hd > lim || a.Wd > lim || a.C > lim || a.N > lim) {
        return hipErrorInvalidValue;
    }
    if (a.N == 0 || a.C == 0) {
        return hipSuccess;
    }
    if (a.x == nullptr || a.y == nullptr) {
        return hipErrorInvalidValue;
    }
    if (a.copy) {
        if (a.elem_in != a.elem_out) {
            return hipErrorInvalidValue;
        }
        return hipMemcpyAsync(a.y, a.x, (size_t)(a.N * a.C * a.Hs * a.Ws) * elem_size(a.elem_in),
                              hipMemcpyDeviceToDevice, stream);
    }
    if (a.elem_in == Elem::F32) {
        switch (a.elem_out) {
            case Elem::F32: return run<float, float>(a, stream);
            case Elem::F16: return run<float, _Float16>(a, stream);
            case Elem::BF16: return run<float, __bf16>(a, stream);
        }
    }
    if (a.elem_in == Elem::F16 && a.elem_out == Elem::F16) {
        return run<_Float16, _Float16>(a, stream);
    }
    if (a.elem_in == Elem::BF16 && a.elem_out == Elem::BF16) {
        return run<__bf16, __bf16>(a, stream);
    }
    return hipErrorInvalidValue;
}

}  // namespace opscv
