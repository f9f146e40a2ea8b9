// Division of indices by a number known at launch (constexpr: for the host and for kernels).
#pragma once

#include <cstdint>

namespace opscv {

// Division of a block index by a launch constant without the hardware's reciprocal sequence (a dependent chain of
// conversions and a reciprocal that every wavefront of the kernel would walk before it knows its work): the host hands
// over m = ceil(2^s / d), s = 31 + ceil(log2 d), and floor(x / d) = (x * m) >> s for every x < 2^31.
struct FastDiv {
    uint32_t mul = 0x80000000u;
    uint32_t shift = 31;
    uint32_t div = 1;
};

inline FastDiv make_fast_div(uint32_t d)
{
    FastDiv f;
    uint32_t l = 0;
    while ((1ull << l) < d) {
        l++;
    }
    f.shift = 31 + l;
    f.mul = (uint32_t)(((1ull << f.shift) + d - 1) / d);
    f.div = d;
    return f;
}

constexpr uint32_t fast_div(uint32_t x, const FastDiv& f)
{
    return (uint32_t)(((uint64_t)x * f.mul) >> f.shift);
}

}  // namespace opscv
