// Which kernel shrinks channels-last images (resize_kernels.hip): host arithmetic only.
#pragma once

#include "acl_types.hpp"

namespace opscv {

// Two output rows together, nothing kept (resize_nhwc_shrink_kernel), or one after the other with kept source rows
// (resize_nhwc_unit_kernel), for units of `unit` bytes of a pixel.
//
// Below a factor of 1.5 most output rows share a source row with the next, and the unit kernel keeps it.  Units of 2 and 6
// bytes, whose loads cost the most per byte, gain from it up to 1.75: pairs against kept rows at 1.5 to 1.6 1.07 and
// 1.11 (medians of 80 images each), 1.6 to 1.7 1.03, 1.7 to 1.8 0.99 and 1.00, at 2 0.93 and 0.95; units of 4 and 12
// bytes 1.01 and 0.97 at 1.5 to 1.6, 0.91 and 0.96 at 2.  Where every output row falls on a source row (whole factors, odd
// ones with half-pixel centres) the unit kernel reads that row alone, half the loads: fp16 1x2160x3840x3 to 720x1280 6.8
// us, 8.9 in pairs, 10x1974x2024x3 to 658x722 22 / 35.
inline bool shrinking_rows_go_in_pairs(const ResizeArgs& a, int unit)
{
    if (!(a.scale_h >= ((unit == 2 || unit == 6) ? 1.75f : 1.5f))) {
        return false;
    }
    const bool on_rows = a.scale_h < 1048576.0f && a.scale_h == (float)(int32_t)a.scale_h &&
                         (a.half_pixel == 0 || ((int32_t)a.scale_h & 1) != 0);
    return !on_rows;
}

}  // namespace opscv
