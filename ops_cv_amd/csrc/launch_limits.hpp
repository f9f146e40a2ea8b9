// What a kernel launch can hold.
#pragma once

#include <cstdint>

namespace opscv {

// Work items of a dispatch along one axis fit 32 bits: from 2^24 workgroups of 256 on a launch is refused.
constexpr bool fits_launch(int64_t blocks, int64_t threads) { return blocks <= (int64_t)UINT32_MAX / threads; }

}  // namespace opscv
