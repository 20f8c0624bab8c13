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

// Tasks of the direct placement: a patch's blocks of 1024 pairs in depth order,
// cut where the work so far (pairs that reach the patch, plus a floor per block)
// passes the next multiple of the aim.
//   aim: a window of 1024 with room for uneven blocks, or more where the patch
//     would have over half of `most` tasks of pairs alone;
//   floor: holds a task to 64 blocks;
//   most: tasks a patch may have, (total + floor blocks) / aim + 1 at most for
//     every total up to 1024 blocks.  The table of counts has 2 KB a task and
//     patch, so it is kept to what the blocks can give: below 448 blocks twice
//     their pairs in units of the aim, which never raises it (10k pairs on 512 x
//     512 tiles: 24 tasks a patch, 25 MB where 384 took 403), then 1024, and from
//     12.8k blocks on a task for every 12.5 of them.
constexpr uint32_t kTaskPairs = 896;
__host__ __device__ inline uint32_t bins_task_aim(uint32_t total, uint32_t most) {
    const uint32_t raised = (uint32_t)(2 * (uint64_t)total / most) + 1;
    return raised > kTaskPairs ? raised : kTaskPairs;
}
__host__ __device__ inline uint32_t bins_block_floor(uint32_t aim) { return aim / 60 + 1; }
__host__ __device__ inline uint32_t bins_most_tasks(uint32_t blocks) {
    const uint32_t all = (uint32_t)(2048ull * blocks / (kTaskPairs - 1)) + 2, many = blocks * 2 / 25;
    const uint32_t few = all < 1024u ? all : 1024u;
    return few > many ? few : many;
}

}  // namespace ubs
