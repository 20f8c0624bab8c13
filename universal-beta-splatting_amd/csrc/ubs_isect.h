// Shared pieces of the tile intersection kernels.
#pragma once

#include "ubs_common.h"

namespace ubs {

// The tile box follows isect_tiles.cu:54-66 exactly: tile_radius and the
// centre are divided by tile_size in fp32, floor/ceil, converted with CUDA's
// saturating float->uint32 semantics and clamped to the grid.
__device__ __forceinline__ void tile_box(float mx, float my, int32_t rad, uint32_t ts, uint32_t tw,
                                         uint32_t th, uint32_t &x0, uint32_t &y0, uint32_t &x1,
                                         uint32_t &y1) {
    const float tr = (float)rad / (float)ts;
    const float tx = mx / (float)ts, ty = my / (float)ts;
    x0 = min(sat_u32(floorf(tx - tr)), tw);
    y0 = min(sat_u32(floorf(ty - tr)), th);
    x1 = min(sat_u32(ceilf(tx + tr)), tw);
    y1 = min(sat_u32(ceilf(ty + tr)), th);
}

}  // namespace ubs
