// Backward of the bilinear resize for gfx950, planes (NCHW): incoming rows in registers, several outgoing rows at a time.
//
// Same visits, products and order of the sum as resize_grad_kernel (resize_grad.hip): an outgoing element visits up to twelve
// rows and columns of the incoming gradient, in row-major order.  A lane owns a column of a plane -- the columns of all planes
// side by side, so that no wavefront is cut by a plane's last column -- and keeps the weights of the columns it visits; a
// wavefront goes down the incoming rows by itself, without barriers.  A row is loaded in aligned units of 16 bytes, three rows
// ahead, passes one or two KB of LDS of the wavefront's own, and every lane reads its run of columns there.  An incoming
// row is visited by two neighbouring outgoing rows: it is read and unpacked once for the sums of both.
//
// Bound by vector instructions, 6 a visited column and pair of rows and some 25 a row: bf16 8x64x65x129 from 257x513 44 us (58
// in the kernel that stages a rectangle for a workgroup, where every outgoing row reads its incoming rows for itself), of which
// 24 are its bytes at the copy rate; fp16 4x16x1080x1920 by two 412 us, 344 of them the issue of 211 M vector instructions.  Runs of columns straight from memory, a load that starts at any element, are 43 us there
// but 46 where rows through LDS take 32 (fp32 4x16x270x480 by two).  Four outgoing rows at a time instead of two as the row
// goes down need branches that cost more than they share.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "fast_div.hpp"
#include "kernels.hpp"
#include "resize_grad_math.hpp"

namespace opscv {

namespace {

constexpr int kActive = 3;  // outgoing rows that are summed together
typedef uint32_t unit_t __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(1))) unit_t* global_unit_t;  // keeps the loads global ones, not flat
constexpr int kAhead = 3;   // incoming rows on their way

// What a wavefront writes to LDS it reads back itself, in order.
__device__ __forceinline__ void wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// TWO: a lane moves up to two 16-byte units of a row, else one.  VISITS: most rows that an element visits (RowsPlan::visits).
template <typename TI, typename TO, bool TWO, int VISITS>
__global__ __launch_bounds__(kGradThreads) void resize_grad_rows_kernel(const TI* __restrict__ g, TO* __restrict__ y,
                                                                         uint32_t columns, FastDiv by_ws, FastDiv by_groups,
                                                                         int32_t rows, uint32_t pieces, int32_t Hs, int32_t Ws,
                                                                         int32_t Hd, int32_t Wd, float scale_h, float scale_w,
                                                                         float inv_scale_h, float inv_scale_w, float offset)
{
    // neighbouring pieces on one XCD: the incoming rows that two groups of outgoing rows visit come from its L2
    constexpr int kTable = 64 / VISITS;  // outgoing rows whose weights the wavefront holds at a time
    const uint32_t piece = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (piece >= pieces) {
        return;
    }
    const uint32_t tile = fast_div(piece, by_groups), group = piece - tile * by_groups.div;
    const int32_t lane = (int32_t)threadIdx.x & 63;
    const uint32_t begin = __builtin_amdgcn_readfirstlane(tile * kGradThreads + (threadIdx.x & ~63u));
    if (begin >= columns) {
        return;
    }
    const bool own = begin + (uint32_t)lane < columns;
    const uint32_t column = own ? begin + (uint32_t)lane : begin;
    const uint32_t plane = fast_div(column, by_ws), plane0 = fast_div(begin, by_ws);
    const int32_t W = (int32_t)(column - plane * (uint32_t)Ws);
    const float fw = (float)W;
    const float last_y = (float)Hs - 1.0f, last_x = (float)Ws - 1.0f;
    const int32_t in_x_start = first_visited(W, inv_scale_w, Wd, offset);
    const float out_x_start = ((float)in_x_start + offset) * scale_w - offset;
    int32_t nx = 0;
    {
        float out_x = out_x_start;
        for (int32_t in_x = in_x_start; out_x < fw + 1.0f && in_x < Wd; in_x++) {
            nx++;
            out_x += scale_w;
        }
    }
    const int32_t H0 = (int32_t)group * rows, H1 = (H0 + rows < Hs) ? H0 + rows : Hs;
    const int64_t in_plane = (int64_t)Hd * Wd;
    __shared__ unit_t s_rows[kGradThreads / 64][64 * (TWO ? 2 : 1) + 3];  // lanes read past their last column
    unit_t* rows_lds = s_rows[threadIdx.x >> 6];
    const TI* g0 = g + (int64_t)plane0 * in_plane;
    TO* y_col = y + (int64_t)plane * Hs * (int64_t)Ws + W;

    // KX: columns read, at least as many as any lane visits.  CUT: some lane visits fewer: the others count as +0, whose
    // products change no sum (a sum is never -0).
    auto sums = [&](auto kx, auto cut) __attribute__((always_inline)) -> bool {
        constexpr int KX = decltype(kx)::value;
        constexpr bool CUT = decltype(cut)::value;
        constexpr int ESZ = (int)sizeof(TI), WORDS = KX * ESZ / 4;
        const int32_t last = Wd > KX ? Wd - KX : 0, from = in_x_start < last ? in_x_start : last, skipped = in_x_start - from;
        float xl[KX];
        uint32_t keep[WORDS];
        {
            float out_x = out_x_start;
#pragma unroll
            for (int k = 0; k < KX; k++) {
                xl[k] = 1.0f - __builtin_fabsf(__builtin_fmaxf(0.0f, __builtin_fminf(out_x, last_x)) - fw);
                out_x = (k >= skipped) ? out_x + scale_w : out_x;
            }
            auto visited = [&](int k) __attribute__((always_inline)) { return k >= skipped && k < skipped + nx; };
#pragma unroll
            for (int i = 0; i < WORDS; i++) {
                if constexpr (sizeof(TI) == 4) {
                    keep[i] = visited(i) ? 0xFFFFFFFFu : 0u;
                } else {
                    keep[i] = (visited(2 * i) ? 0xFFFFu : 0u) | (visited(2 * i + 1) ? 0xFFFF0000u : 0u);
                }
            }
        }
        // A row of the wavefront's columns as 16-byte units, a lane each, plane after plane: of the first plane the run that its
        // columns visit, of the others from the row's first element on.  A unit has at least one byte of its run, so that it
        // is readable; past the run's last one a lane loads that again.  Offsets are from an aligned address of the wavefront.
        const int32_t lanes = (columns - begin < 64u) ? (int32_t)(columns - begin) : 64;
        const int32_t W_first = __builtin_amdgcn_readfirstlane(W), lanes0 = (Ws - W_first < lanes) ? Ws - W_first : lanes;
        const int32_t from0 = __builtin_amdgcn_readlane(from, 0);
        auto run_end = [&](int32_t of) __attribute__((always_inline)) {
            const int32_t end = __builtin_amdgcn_readlane(from, of) + KX;
            return end < Wd ? end : Wd;
        };
        const int32_t bytes0 = (run_end(lanes0 - 1) - from0) * ESZ;
        const int32_t planes_whole = lanes0 < lanes ? (lanes - lanes0) / Ws : 0, lanes_last = (lanes - lanes0) - planes_whole * Ws;
        const int32_t bytes_last = lanes_last > 0 ? run_end(lanes - 1) * ESZ : 0;
        const int32_t units0 = (bytes0 + 30) >> 4, units = (Wd * ESZ + 30) >> 4, units_last = lanes_last > 0 ? (bytes_last + 30) >> 4 : 0;
        const int32_t units_all = units0 + planes_whole * units + units_last;
        if (units_all > (TWO ? 128 : 64)) {
            return false;
        }
        const uintptr_t aligned = reinterpret_cast<uintptr_t>(g0 + from0) & ~(uintptr_t)15;
        const uint32_t low = (uint32_t)(reinterpret_cast<uintptr_t>(g0 + from0) & 15u);
        const uint32_t pitch = (uint32_t)Wd * (uint32_t)ESZ, plane_bytes = (uint32_t)in_plane * (uint32_t)ESZ;
        // of the plane'th plane of the wavefront: where its run begins
        auto run_of = [&](int32_t i) __attribute__((always_inline)) { return low + (uint32_t)i * plane_bytes - (i > 0 ? (uint32_t)(from0 * ESZ) : 0u); };
        uint32_t unit_at[2];
#pragma unroll
        for (int n = 0; n < (TWO ? 2 : 1); n++) {
            const int32_t u = n * 64 + lane < units_all ? n * 64 + lane : units_all - 1;
            int32_t i = 0, k = u;
            if (lanes0 < lanes && u >= units0) {
                i = 1 + (u - units0) / units;
                k = u - units0 - (i - 1) * units;
            }
            const int32_t bytes = i == 0 ? bytes0 : (i > planes_whole ? bytes_last : Wd * ESZ);
            const uint32_t begins = run_of(i), last = begins + (uint32_t)bytes - 1u, own_unit = begins + (uint32_t)k * 16u;
            unit_at[n] = own_unit < last ? own_unit : last;
        }
        const int32_t my = (int32_t)(plane - plane0);
        const uint32_t my_run = run_of(my), my_units = (uint32_t)(my == 0 ? 0 : units0 + (my - 1) * units) * 16u;
        const uint32_t my_first = (uint32_t)(from - (my == 0 ? from0 : 0)) * (uint32_t)ESZ;

        // The rows that outgoing rows from `base` on visit and their weights, a lane each: lane VISITS q + j the j-th of row
        // base + q.  False: one visits more.
        int32_t base = H0, start = 0;
        float weight = 0.0f;
        uint64_t visited_rows = 0;
        auto table = [&]() __attribute__((always_inline)) {
            const int32_t q = lane / VISITS, j = lane - q * VISITS, H = base + q;
            start = first_visited(H, inv_scale_h, Hd, offset);
            const float fh = (float)H;
            float out_y = ((float)start + offset) * scale_h - offset;
#pragma unroll
            for (int u = 0; u < VISITS - 1; u++) {
                out_y = (u < j) ? out_y + scale_h : out_y;
            }
            weight = 1.0f - __builtin_fabsf(__builtin_amdgcn_fmed3f(out_y, 0.0f, last_y) - fh);
            const bool visits = q < kTable && H < H1 && out_y < fh + 1.0f && start + j < Hd;
            visited_rows = __builtin_amdgcn_ballot_w64(visits);
            const bool beyond = j == VISITS - 1 && visits && out_y + scale_h < fh + 1.0f && start + VISITS < Hd;
            return __builtin_amdgcn_ballot_w64(beyond) == 0ull;
        };
        auto first_of = [&](int32_t H) __attribute__((always_inline)) { return H < H1 ? __builtin_amdgcn_readlane(start, (H - base) * VISITS) : INT32_MAX; };
        auto end_of = [&](int32_t H, int32_t first) __attribute__((always_inline)) {
            return H < H1 ? first + __builtin_popcount((uint32_t)(visited_rows >> ((H - base) * VISITS)) & ((1u << VISITS) - 1u)) : INT32_MAX;
        };
        // Down the incoming rows: row r goes to the sums of the outgoing rows that visit it, H, H + 1 and, where rounding has
        // an integer coordinate on both sides, H + 2.  H is done when r is behind its last row.
        int32_t H = H0;
        if (!table()) {
            return false;
        }
        int32_t first[kActive], end0;
        float acc[kActive];
#pragma unroll
        for (int i = 0; i < kActive; i++) {
            first[i] = first_of(H + i);
            acc[i] = 0.0f;
        }
        end0 = end_of(H, first[0]);
        int32_t r = first[0], slot = 0;  // slot: VISITS (H - base)
        struct Row {  // a lane's units of an incoming row
            unit_t a, b;
        };
        auto load = [&](int32_t row) __attribute__((always_inline)) {
            const uint32_t at = (uint32_t)(row < Hd ? row : Hd - 1) * pitch;
            Row w;
            w.a = *(global_unit_t)(aligned + ((unit_at[0] + at) & ~15u));
            if constexpr (TWO) {
                w.b = *(global_unit_t)(aligned + ((unit_at[1] + at) & ~15u));
            }
            return w;
        };
        auto step = [&](Row& row) __attribute__((always_inline)) {
                rows_lds[lane] = row.a;
                if constexpr (TWO) {
                    rows_lds[64 + lane] = row.b;
                }
                row = load(r + kAhead);
                wave_fence();
                const uint32_t at = my_units + my_first + ((my_run + (uint32_t)r * pitch) & 15u);
                const uint32_t* words = reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(rows_lds) + (at & ~3u));
                uint32_t w[WORDS + 1];
#pragma unroll
                for (int i = 0; i < WORDS + (ESZ == 2 ? 1 : 0); i++) {
                    w[i] = words[i];
                }
                wave_fence();
                float f[KX];
#pragma unroll
                for (int i = 0; i < WORDS; i++) {
                    // 16-bit pairs are shifted into place: alignbit takes the low five bits, 0 or 16
                    uint32_t bits = (ESZ == 2) ? __builtin_amdgcn_alignbit(w[i + 1], w[i], at << 3) : w[i];
                    if constexpr (CUT) {
                        bits &= keep[i];
                    }
                    TI v[4 / ESZ];
                    __builtin_memcpy(v, &bits, 4);
#pragma unroll
                    for (int k = 0; k < 4 / ESZ; k++) {
                        f[i * (4 / ESZ) + k] = ElemIO<TI>::load(&v[k]);
                    }
                }
                auto add = [&](int i) __attribute__((always_inline)) {
                    const float y_lerp = __builtin_bit_cast(
                        float, __builtin_amdgcn_readlane(__builtin_bit_cast(int32_t, weight), slot + i * VISITS + r - first[i]));
#pragma unroll
                    for (int k = 0; k < KX; k++) {
                        acc[i] += f[k] * y_lerp * xl[k];
                    }
                };
                if (r >= first[0]) {
                    add(0);
                }
                if (r >= first[1]) {
                    add(1);
                    if (r >= first[2]) {
                        add(2);
                    }
                }
                r++;
        };
        auto store = [&]() __attribute__((always_inline)) {
            if (own) {
                store_streaming<TO>(y_col + (int64_t)H * Ws, acc[0]);
            }
            H++;
        };
        auto next = [&]() __attribute__((always_inline)) {
            slot = (H - base) * VISITS;
#pragma unroll
            for (int i = 0; i + 1 < kActive; i++) {
                first[i] = first[i + 1];
                acc[i] = acc[i + 1];
            }
            first[kActive - 1] = first_of(H + kActive - 1);
            acc[kActive - 1] = 0.0f;
            end0 = end_of(H, first[0]);
        };
        Row one = load(r);
        __builtin_amdgcn_sched_barrier(0);  // in this order, as in the loop
        Row two = load(r + 1);
        __builtin_amdgcn_sched_barrier(0);
        Row three = load(r + 2);
        __builtin_amdgcn_sched_barrier(0);
        // jumps out of the loop rather than flags, which would hide from the compiler how many loads are on their way
#define OPSCV_STEP(ROW)                                                  \
    while (r >= end0) {                                                  \
        store();                                                         \
        if (H >= H1) {                                                   \
            goto finished;                                               \
        }                                                                \
        if (H + kActive > base + kTable && base + kTable < H1) { \
            base = H;                                                    \
            if (!table()) {                                              \
                goto refused;                                            \
            }                                                            \
        }                                                                \
        next();                                                          \
    }                                                                    \
    step(ROW);
        for (;;) {
            OPSCV_STEP(one)
            OPSCV_STEP(two)
            OPSCV_STEP(three)
        }
#undef OPSCV_STEP
    finished:
        return true;
    refused:
        return false;
    };
    auto any = [&](bool b) __attribute__((always_inline)) { return __builtin_amdgcn_ballot_w64(b) != 0ull; };
    auto width = [&](auto kx) __attribute__((always_inline)) {
        return any(nx < decltype(kx)::value) ? sums(kx, std::true_type{}) : sums(kx, std::false_type{});
    };
    bool done = false;
    if (any(nx > (VISITS == kRowsColumns ? kRowsColumns : 10))) {
    } else if (VISITS == kRowsColumns && any(nx > 10)) {
        done = width(std::integral_constant<int, VISITS == kRowsColumns ? kRowsColumns : 10>{});
    } else if (any(nx > 8)) {
        done = width(std::integral_constant<int, 10>{});
    } else if (any(nx > 6)) {
        done = width(std::integral_constant<int, 8>{});
    } else if (any(nx > 4)) {
        done = width(std::integral_constant<int, 6>{});
    } else if (any(nx > 2)) {
        done = width(std::integral_constant<int, 4>{});
    } else {
        done = width(std::integral_constant<int, 2>{});
    }
    if (!done) {  // an element visits more rows or columns
        for (int32_t r = H0; own && r < H1; r++) {
            const int32_t in_y_start = first_visited(r, inv_scale_h, Hd, offset);
            store_streaming<TO>(y_col + (int64_t)r * Ws,
                                visit_sum<TI>(g + (int64_t)plane * in_plane, Wd, 0, 0, in_y_start, in_x_start,
                                              ((float)in_y_start + offset) * scale_h - offset, out_x_start, (float)r, fw,
                                              scale_h, scale_w, last_y, last_x, Hd, Wd));
        }
    }
}

template <typename TI, typename TO>
hipError_t run_typed(const ResizeGradArgs& a, const RowsPlan& p, hipStream_t stream)
{
    const uint32_t tiles = (p.columns + kGradThreads - 1) / kGradThreads;
#define OPSCV_RGR(TWO, VISITS)                                                                                               \
    hipLaunchKernelGGL((resize_grad_rows_kernel<TI, TO, TWO, VISITS>), dim3((unsigned)p.blocks), dim3(kGradThreads), 0,      \
                       stream, (const TI*)a.x, (TO*)a.y, p.columns, p.by_ws, p.by_groups, p.rows, tiles * p.by_groups.div,   \
                       (int32_t)a.Hs, (int32_t)a.Ws, (int32_t)a.Hd, (int32_t)a.Wd, a.scale_h, a.scale_w, a.inv_scale_h,      \
                       a.inv_scale_w, a.half_pixel ? 0.5f : 0.0f)
    if (p.two) {
        switch (p.visits) {
            case kRowsColumns: OPSCV_RGR(true, kRowsColumns); break;
            case 10: OPSCV_RGR(true, 10); break;
            default: OPSCV_RGR(true, 8); break;
        }
    } else {
        switch (p.visits) {
            case kRowsColumns: OPSCV_RGR(false, kRowsColumns); break;
            case 10: OPSCV_RGR(false, 10); break;
            default: OPSCV_RGR(false, 8); break;
        }
    }
#undef OPSCV_RGR
    return hipGetLastError();
}

}  // namespace

hipError_t run_resize_grad_rows(const ResizeGradArgs& a, const RowsPlan& p, hipStream_t stream)
{
    if (a.elem_in == Elem::F32) {
        switch (a.elem_out) {
            case Elem::F32: return run_typed<float, float>(a, p, stream);
            case Elem::F16: return run_typed<float, _Float16>(a, p, stream);
            case Elem::BF16: return run_typed<float, __bf16>(a, p, stream);
        }
    }
    if (a.elem_in == Elem::F16 && a.elem_out == Elem::F16) {
        return run_typed<_Float16, _Float16>(a, p, stream);
    }
    if (a.elem_in == Elem::BF16 && a.elem_out == Elem::BF16) {
        return run_typed<__bf16, __bf16>(a, p, stream);
    }
    return hipErrorInvalidValue;
}

}  // namespace opscv
