// Input gradient of the samplers as a gather over sorted contribution lists (gs_grad_gather.hip): what the launchers of
// the 2-D and 3-D backward hand over.
#pragma once

#include <hip/hip_runtime_api.h>

#include "gs_grad_gather_plan.hpp"

namespace opscv {

// 32-bit words of scratch, 0 where the shape is beyond what the kernels index
int64_t grad_gather_words(const GradGatherArgs& a);
hipError_t run_grad_gather(const GradGatherArgs& a, hipStream_t stream, bool* dgrid_done);  // sets *dgrid_done where it was taken along

// the same by tiles of the plane or volume (gs_grad_tiles.hip)
int64_t grad_tiles_words(const GradGatherArgs& a);
hipError_t run_grad_tiles(const GradGatherArgs& a, hipStream_t stream, bool* dgrid_done);

}  // namespace opscv
