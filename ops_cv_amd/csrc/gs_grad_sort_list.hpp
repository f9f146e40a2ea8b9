// A lane's list of contribution keys sorted through registers (gs3d_grad_lists.hip, gs_grad_gather.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace opscv {

// The first NK entries of a lane's list (every STRIDE-th word from `mine`), sorted ascending by a bitonic network; past its
// end the list is padded with the largest key.
template <int NK, int STRIDE>
__device__ __forceinline__ void sort_list(uint32_t* mine, uint32_t len)
{
    uint32_t key[NK];
#pragma unroll
    for (int i = 0; i < NK; i++) {
        const uint32_t v = mine[i * STRIDE];
        key[i] = ((uint32_t)i < len) ? v : 0xFFFFFFFFu;
    }
#pragma unroll
    for (int size = 2; size <= NK; size *= 2) {
#pragma unroll
        for (int stride = size / 2; stride > 0; stride /= 2) {
#pragma unroll
            for (int i = 0; i < NK; i++) {
                const int l = i ^ stride;
                if (l > i) {
                    const uint32_t lo = key[i] < key[l] ? key[i] : key[l];
                    const uint32_t hi = key[i] < key[l] ? key[l] : key[i];
                    const bool ascending = (i & size) == 0;
                    key[i] = ascending ? lo : hi;
                    key[l] = ascending ? hi : lo;
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < NK; i++) {
        mine[i * STRIDE] = key[i];
    }
}

}  // namespace opscv
