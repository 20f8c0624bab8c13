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

// Whether placing the entries beats emitting and sorting them: 1 yes, 0 no, or,
// with n_isects unknown (-1), 2: it depends on it.  Measured on both ways, us (1 to 8
// cameras of 10k to 1M pairs, 1 x 1 to 512 x 512 tiles, all to 1% of them visible):
//   - the sort moves an entry five times, 15 a million entries; its offset search
//     runs over the tiles between two entries, 2.9 for every tile per entry; its
//     launches 52 in all;
//   - the placement looks at every patch for every pair and at its tiles one
//     patch after another: 0.72 a patch and 0.21 a patch and million pairs.
// 512 x 512 tiles (512 patches), 1M pairs, 5.9M entries: placed 872, sorted 465; 8
// views of 1080p (136 patches), 8M pairs, 0.46M entries 1028 and 746, 46M entries 1834
// and 2295; 616 entries on 512 x 512 tiles 530 and 1303.
// A tile's entries of a window are stored by 16 lanes, so few tiles leave the chip
// idle (1 x 1 tiles, 1M pairs: 430 placed, 249 sorted; 2 x 2: 331 and 282; 4 x 4 and
// 100k: 188 and 182; 8 x 8: 177 and 187).
constexpr uint32_t kPlaceMinTiles = 32;
inline int bins_pays(uint64_t pairs, uint64_t tiles, uint32_t patches, int64_t n_isects) {
    if (tiles < kPlaceMinTiles) return 0;
    const double place = patches * (0.72 + 0.21e-6 * (double)pairs);
    if (place <= 52.0) return 1;
    if (n_isects < 0) return 2;
    const double n = n_isects > 0 ? (double)n_isects : 1.0;
    return place <= 52.0 + 15e-6 * n + 2.9 * (double)tiles / n;
}

}  // namespace ubs
