// Input gradient of the samplers as a gather over sorted contribution lists (gs_grad_gather.hip): what the launchers of
// the 2-D and 3-D backward hand over.
#pragma once

#include <hip/hip_runtime_api.h>

#include "acl_types.hpp"

namespace opscv {

constexpr int64_t kGatherMaxScratch = (int64_t)4 << 30;  // bytes of a call, of the 288 GB of the device

struct GradGatherArgs {
    Elem elem = Elem::F32;
    int dim = 2;
    int interp = 0, pad = 0, align = 0;
    int64_t N = 0, C = 0, D = 1, H = 0, W = 0;
    int64_t points = 0;          // grid points per batch item
    int64_t items_per_core = 1;  // batch items whose points are cut into chunks as one run (3-D; 1 for planes)
    const void* gout = nullptr;
    const void* grid = nullptr;
    void* dx = nullptr;
    void* scratch = nullptr;  // grad_gather_words() 32-bit words on a 16-byte boundary
};

// 32-bit words of scratch, 0 where the shape is beyond what the kernels index
int64_t grad_gather_words(const GradGatherArgs& a);
hipError_t run_grad_gather(const GradGatherArgs& a, hipStream_t stream);

}  // namespace opscv
