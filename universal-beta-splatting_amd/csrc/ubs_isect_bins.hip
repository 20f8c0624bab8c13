// Tile lists by direct placement on gfx950: from the (camera, primitive)
// pairs in depth order to the sorted intersection list in one write.
//
// A sort of the emitted entries on their camera/tile bits moves 12 bytes an
// entry five times (emission, two passes that read and write) and reads the keys
// twice more.  The place of an entry is known without moving it: its tile's
// start, plus the tile's entries of earlier pairs.  The grid of tiles (the
// cameras' grids stacked: row = camera * th + ty) is cut into patches of 32 x 16
// tiles:
//   pairs    each pair's record in depth order (id, depth, tile box), and per
//            patch one bit a pair: its box reaches the patch;
//   cuts     per patch: the depth order cut into tasks of about equal numbers of
//            pairs that reach it (most patches meet them at some depths only, and
//            a task of many pairs with large boxes is the tail of the launch);
//   count    per task: entries of each tile, from the corners of the boxes summed
//            over both axes;
//   rows     per tile: the counts' running sum over its patch's tasks;
//   offsets  running sum over the tiles: the tile lists' starts;
//   place    per task: the pairs that reach the patch, 1024 at a time, as
//            one bit a pair in each column and each row of the patch; the
//            entries of tile (x, y) are the set bits of column x AND row y, in
//            depth order.  16 lanes take a tile: a lane a word of 64 pairs,
//            a prefix sum of the popcounts, the pairs' numbers gathered in LDS
//            and stored by consecutive lanes.
// No atomics on memory, no look-back: the result does not depend on the order
// in which anything runs.
//
// 13.8 M entries of 1M pairs at 1080p: 151 us in all (pairs 28, cuts 5, count 21,
// rows 6, offsets 9, place 82) against 403 for emission, the two sort passes with
// their histograms and the offsets.  Place is bound by the latency of a tile's LDS
// steps and the stores of short runs (a window has about 20 entries of a tile; the
// 166 MB alone take 31 us).  Half-waves per tile over windows of 32 x 32 tiles:
// 156 us on evenly spread pairs (74 now); tasks of equal numbers of pairs in depth
// order, whatever patch: 132-174 (the tail); 256 threads: 80-94, 1024: 115.
#pragma clang fp contract(off)

#include "ubs_common.h"
#include "ubs_isect.h"

namespace ubs {

constexpr uint32_t kPatchX = 32, kPatchY = 16;        // tiles of a patch
constexpr uint32_t kPatchTiles = kPatchX * kPatchY;
constexpr uint32_t kWindow = 1024;                    // pairs placed together
constexpr uint32_t kTileLanes = 16;                   // lanes per tile: a word of 64 pairs each
constexpr uint32_t kPlaceThreads = 512;
constexpr uint32_t kStage = 64;                       // entries of a tile gathered in LDS before they are stored
constexpr uint32_t kPairGroups = 16;                  // groups of 64 pairs of a block: the pairs kernel's workgroup, the unit of a cut
constexpr uint32_t kPairPatches = 32;                 // patches whose bits it writes together
constexpr uint32_t kTaskWords = 4;                    // groups of a task per thread of count (of kThreads), at most
constexpr uint32_t kMaxPatches = 512;
// Workgroups of count and place (fewer where there are fewer tasks): more than are
// resident, so that what is left over at the end is small.
constexpr uint32_t kCountBlocks = 2048, kPlaceBlocks = 4096;

struct BinShape {
    uint32_t px, py, patches;   // patches of the stacked tile grid
    uint32_t groups, most;      // groups of 64 pairs (padded to the pairs kernel's), most tasks of a patch
    uint64_t bins;
    size_t bits, sums, cuts, tasks, counts, totals, bytes;  // offsets into the workspace (records at 0) and its size
};

// false: grids or counts past the packed fields; the sort serves those.
static bool bin_shape(uint32_t C, uint32_t N, uint32_t tw, uint32_t th, BinShape &s) {
    const uint64_t total = (uint64_t)C * N, rows = (uint64_t)C * th;
    if (total == 0 || total >= (1ull << 31) || tw == 0 || rows == 0 || tw > 0xFFFFu || rows > 0xFFFFu) return false;
    s.px = (tw + kPatchX - 1) / kPatchX;
    s.py = ((uint32_t)rows + kPatchY - 1) / kPatchY;
    if ((uint64_t)s.px * s.py > kMaxPatches) return false;
    s.patches = s.px * s.py;
    s.groups = (uint32_t)((total + 64 * kPairGroups - 1) / (64 * kPairGroups)) * kPairGroups;
    s.most = bins_most_tasks(s.groups / kPairGroups);
    s.bins = (uint64_t)tw * rows;
    auto up = [](size_t v) { return (v + 255) & ~(size_t)255; };
    s.bits = up((size_t)total * sizeof(uint4));
    s.sums = s.bits + up((size_t)s.patches * s.groups * sizeof(uint64_t));
    s.cuts = s.sums + up((size_t)s.patches * (s.groups / kPairGroups) * sizeof(uint32_t));
    s.tasks = s.cuts + up((size_t)s.patches * (s.most + 1) * sizeof(uint32_t));
    s.counts = s.tasks + up((size_t)s.patches * sizeof(uint32_t));
    s.totals = s.counts + up((size_t)s.patches * s.most * kPatchTiles * sizeof(uint32_t));
    s.bytes = s.totals + up((size_t)s.bins * sizeof(uint32_t));
    return true;
}

// records[k]: of the pair at place k of the depth order: (flat id, depth bits,
// x0 | x1 << 16, row0 | row1 << 16), the box empty for a culled pair (or an order
// entry outside [0, C N), only from a depth sort that gave up).
__global__ __launch_bounds__(kThreads) void bins_pairs_kernel(uint32_t total, uint32_t N, const float4 *__restrict__ prec,
                                                              const int32_t *__restrict__ order, uint32_t ts,
                                                              uint32_t tw, uint32_t th, uint32_t px, uint32_t patches,
                                                              uint32_t groups, uint4 *__restrict__ records,
                                                              uint64_t *__restrict__ bits,
                                                              uint32_t *__restrict__ sums) {
    constexpr uint32_t kPer = kPairGroups / (kThreads / 64);  // groups per wave
    __shared__ uint64_t s_bits[kPairPatches][kPairGroups];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t g0 = blockIdx.x * kPairGroups + wave * kPer;
    uint32_t idx[kPer];
    float4 pr[kPer];
#pragma unroll
    for (uint32_t u = 0; u < kPer; ++u) {
        const uint32_t k = (g0 + u) * 64 + lane;
        idx[u] = k < total ? (uint32_t)order[k] : total;
    }
#pragma unroll
    for (uint32_t u = 0; u < kPer; ++u)
        pr[u] = idx[u] < total ? prec[idx[u]] : make_float4(0.f, 0.f, 0.f, 0.f);
    uint32_t cx0[kPer], cx1[kPer], cy0[kPer], cy1[kPer];  // the patches the box reaches: [c0, c1]
#pragma unroll
    for (uint32_t u = 0; u < kPer; ++u) {
        uint32_t x0 = 0, y0 = 0, x1 = 0, y1 = 0;
        const int32_t r = __float_as_int(pr[u].z);
        if (r > 0) tile_box(pr[u].x, pr[u].y, r, ts, tw, th, x0, y0, x1, y1);
        if (x0 >= x1 || y0 >= y1) x0 = y0 = x1 = y1 = 0;
        const uint32_t row = x1 ? idx[u] / N * th : 0u;
        y0 += row;
        y1 += row;
        const uint32_t k = (g0 + u) * 64 + lane;
        if (k < total) records[k] = make_uint4(idx[u], __float_as_uint(pr[u].w), x0 | x1 << 16, y0 | y1 << 16);
        cx0[u] = x1 ? x0 / kPatchX : 1u;  // (an empty box: an empty range)
        cx1[u] = x1 ? (x1 - 1) / kPatchX : 0u;
        cy0[u] = y0 / kPatchY;
        cy1[u] = x1 ? (y1 - 1) / kPatchY : 0u;
    }
    uint32_t pc = 0, prow = 0;  // patch column and row
    for (uint32_t p0 = 0; p0 < patches; p0 += kPairPatches) {
        const uint32_t pn = min(kPairPatches, patches - p0);
        for (uint32_t p = 0; p < pn; ++p) {
#pragma unroll
            for (uint32_t u = 0; u < kPer; ++u) {
                const uint64_t b = __ballot(cx0[u] <= pc && pc <= cx1[u] && cy0[u] <= prow && prow <= cy1[u]);
                if (lane == 0) s_bits[p][wave * kPer + u] = b;
            }
            if (++pc == px) {
                pc = 0;
                ++prow;
            }
        }
        __syncthreads();
        for (uint32_t q = threadIdx.x; q < pn * kPairGroups; q += kThreads)
            bits[(size_t)(p0 + q / kPairGroups) * groups + blockIdx.x * kPairGroups + q % kPairGroups] =
                s_bits[q / kPairGroups][q % kPairGroups];
        if (threadIdx.x < pn) {  // the block's pairs that reach the patch
            uint32_t n = 0;
#pragma unroll
            for (uint32_t u = 0; u < kPairGroups; ++u) n += (uint32_t)__popcll(s_bits[threadIdx.x][u]);
            sums[(size_t)(p0 + threadIdx.x) * gridDim.x + blockIdx.x] = n;
        }
        __syncthreads();
    }
}

// cuts[patch][k], k = 0 .. tasks[patch]: the first block of the patch's task k.  A
// block's work is its number of pairs that reach the patch, plus a floor that
// holds a task to 64 blocks; a task ends where the work so far reaches its next
// multiple of the aim.  The aim is kTaskPairs, or more where the patch would have
// more than half of `most` tasks.  One workgroup per patch.
constexpr uint32_t kCutThreads = 1024;
__global__ __launch_bounds__(kCutThreads) void bins_cuts_kernel(uint32_t blocks, uint32_t most,
                                                                const uint32_t *__restrict__ sums,
                                                                uint32_t *__restrict__ cuts,
                                                                uint32_t *__restrict__ tasks) {
    constexpr uint32_t U = 8, kWaves = kCutThreads / 64;
    __shared__ uint32_t s_wave[kWaves];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t *const w = sums + (size_t)blockIdx.x * blocks;
    uint32_t *const cut = cuts + (size_t)blockIdx.x * (most + 1);
    // each thread its own run of blocks
    const uint32_t per = (blocks + kCutThreads - 1) / kCutThreads;
    const uint32_t g0 = min(threadIdx.x * per, blocks), g1 = min(g0 + per, blocks);
    uint32_t own = 0;
    for (uint32_t g = g0; g < g1; g += U) {
        uint32_t v[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) v[u] = g + u < g1 ? w[g + u] : 0u;
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) own += v[u];
    }
    uint32_t inc = own;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t x = __shfl_up(inc, o, 64);
        if ((int)lane >= o) inc += x;
    }
    if (lane == 63) s_wave[wave] = inc;
    __syncthreads();
    uint32_t at = inc - own, total = 0;
    for (uint32_t q = 0; q < kWaves; ++q) {
        at += q < wave ? s_wave[q] : 0u;
        total += s_wave[q];
    }
    const uint32_t aim = bins_task_aim(total, most), floor = bins_block_floor(aim);
    at += floor * g0;
    uint32_t k = at / aim;
    for (uint32_t g = g0; g < g1; g += U) {
        uint32_t v[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) v[u] = g + u < g1 ? w[g + u] : 0u;
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            if (g + u >= g1) break;
            at += v[u] + floor;
            // (a block of more work than the aim may end two: the second is empty)
            for (const uint32_t e = at / aim; k < e;) cut[++k] = g + u + 1;
        }
    }
    if (threadIdx.x == 0) {
        const uint32_t ends = (total + floor * blocks) / aim;
        cut[0] = 0;
        cut[ends + 1] = blocks;
        tasks[blockIdx.x] = ends + 1;
    }
}

// The pairs of one task: each thread holds up to
// kTaskWords of the task's bit words and the number of set bits before them.
template <uint32_t THREADS>
struct TaskBits {
    uint64_t w[kTaskWords];
    uint32_t first;         // group of w[0]
    uint32_t start, total;  // set bits before w[0], and in the task
    __device__ __forceinline__ void load(const uint64_t *__restrict__ bits, uint32_t g0, uint32_t g1, uint32_t *s_wave) {
        const uint32_t per = (g1 - g0 + THREADS - 1) / THREADS;  // <= kTaskWords
        first = g0 + threadIdx.x * per;
        uint32_t n = 0;
#pragma unroll
        for (uint32_t u = 0; u < kTaskWords; ++u) {
            w[u] = u < per && first + u < g1 ? bits[first + u] : 0ull;
            n += (uint32_t)__popcll(w[u]);
        }
        uint32_t inc = n;
        const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t v = __shfl_up(inc, o, 64);
            if ((int)lane >= o) inc += v;
        }
        if (lane == 63) s_wave[wave] = inc;
        __syncthreads();
        uint32_t before = 0;
        total = 0;
#pragma unroll
        for (uint32_t q = 0; q < THREADS / 64; ++q) {
            const uint32_t v = s_wave[q];
            before += q < wave ? v : 0u;
            total += v;
        }
        start = before + inc - n;
    }
    // places [lo, lo + kWindow) of the set bits, as places of the depth order
    __device__ __forceinline__ void window(uint32_t lo, uint32_t *s_list) const {
        uint32_t at = start;
#pragma unroll
        for (uint32_t u = 0; u < kTaskWords; ++u) {
            uint64_t m = w[u];
            const uint32_t n = (uint32_t)__popcll(m);
            if (at + n <= lo || at >= lo + kWindow) {  // (none of them in the window)
                at += n;
                continue;
            }
            while (m) {
                if (at - lo < kWindow) s_list[at - lo] = (first + u) * 64 + (uint32_t)__builtin_ctzll(m);
                m &= m - 1;
                ++at;
            }
        }
    }
};

// All tasks, patch by patch.  A grid of count or place takes every gridDim.x-th
// (how many there are is known on the device only).
template <uint32_t THREADS>
struct Tasks {
    static constexpr uint32_t kPer = kMaxPatches / THREADS;  // patches per thread
    uint32_t total;
    __device__ __forceinline__ void load(const uint32_t *__restrict__ tasks, uint32_t patches, uint32_t *s_first,
                                         uint32_t *s_wave) {
        const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        uint32_t c[kPer], n = 0;
#pragma unroll
        for (uint32_t u = 0; u < kPer; ++u) {
            const uint32_t p = threadIdx.x * kPer + u;
            c[u] = p < patches ? tasks[p] : 0u;
            n += c[u];
        }
        uint32_t inc = n;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t v = __shfl_up(inc, o, 64);
            if ((int)lane >= o) inc += v;
        }
        if (lane == 63) s_wave[wave] = inc;
        __syncthreads();
        uint32_t at = inc - n;
        total = 0;
#pragma unroll
        for (uint32_t q = 0; q < THREADS / 64; ++q) {
            at += q < wave ? s_wave[q] : 0u;
            total += s_wave[q];
        }
#pragma unroll
        for (uint32_t u = 0; u < kPer; ++u) {
            s_first[threadIdx.x * kPer + u] = at;
            at += c[u];
        }
        __syncthreads();
    }
    // the patch of a task below total: the last whose first task is at most it
    __device__ __forceinline__ static uint32_t patch(uint32_t task, const uint32_t *s_first) {
        uint32_t p = 0;
#pragma unroll
        for (uint32_t d = kMaxPatches / 2; d >= 1; d >>= 1)
            if (s_first[p + d] <= task) p += d;
        return (uint32_t)__builtin_amdgcn_readfirstlane((int)p);
    }
};

// The part of a record's box inside the patch at (bx, by), relative to it.
struct PatchBox {
    uint32_t x0, x1, y0, y1;
    __device__ __forceinline__ PatchBox(uint32_t xs, uint32_t ys, uint32_t bx, uint32_t by) {
        x0 = max(xs & 0xFFFFu, bx) - bx;
        x1 = min(xs >> 16, bx + kPatchX) - bx;
        y0 = max(ys & 0xFFFFu, by) - by;
        y1 = min(ys >> 16, by + kPatchY) - by;
    }
};

// counts[patch][task][tile of the patch].  A box adds 1 over itself: four
// corners, then the sums along both axes.
__global__ __launch_bounds__(kThreads) void bins_count_kernel(uint32_t tw, uint32_t rows, uint32_t px, uint32_t patches,
                                                              uint32_t groups, uint32_t most,
                                                              const uint32_t *__restrict__ cuts,
                                                              const uint32_t *__restrict__ tasks,
                                                              const uint4 *__restrict__ records,
                                                              const uint64_t *__restrict__ bits,
                                                              uint32_t *__restrict__ counts) {
    constexpr uint32_t kPitch = kPatchX + 1;  // (33: the sums down a column and along a row miss each other's banks)
    __shared__ int32_t s_sum[kPitch * (kPatchY + 1)];
    __shared__ uint32_t s_list[kWindow];
    __shared__ uint32_t s_first[kMaxPatches];
    __shared__ uint32_t s_wave[kThreads / 64];
    Tasks<kThreads> all;
    all.load(tasks, patches, s_first, s_wave);
    for (uint32_t task = blockIdx.x; task < all.total; task += gridDim.x) {
        const uint32_t p = all.patch(task, s_first), k0 = task - s_first[p];
        const uint32_t *const cut = cuts + (size_t)p * (most + 1) + k0;
        const uint32_t bx = p % px * kPatchX, by = p / px * kPatchY;
        for (uint32_t q = threadIdx.x; q < kPitch * (kPatchY + 1); q += kThreads) s_sum[q] = 0;
        TaskBits<kThreads> sb;
        sb.load(bits + (size_t)p * groups, cut[0] * kPairGroups, cut[1] * kPairGroups, s_wave);
        for (uint32_t lo = 0; lo < sb.total; lo += kWindow) {
            __syncthreads();
            sb.window(lo, s_list);
            __syncthreads();
            const uint32_t n = min(kWindow, sb.total - lo);
            for (uint32_t i = threadIdx.x; i < n; i += kThreads) {
                const uint2 box = reinterpret_cast<const uint2 *>(records + s_list[i])[1];
                const PatchBox q(box.x, box.y, bx, by);
                atomicAdd(&s_sum[q.y0 * kPitch + q.x0], 1);
                atomicAdd(&s_sum[q.y0 * kPitch + q.x1], -1);
                atomicAdd(&s_sum[q.y1 * kPitch + q.x0], -1);
                atomicAdd(&s_sum[q.y1 * kPitch + q.x1], 1);
            }
        }
        __syncthreads();
        if (threadIdx.x < kPatchY) {
            int32_t run = 0;
            for (uint32_t x = 0; x < kPatchX; ++x)
                s_sum[threadIdx.x * kPitch + x] = run += s_sum[threadIdx.x * kPitch + x];
        }
        __syncthreads();
        if (threadIdx.x < kPatchX) {
            int32_t run = 0;
            for (uint32_t y = 0; y < kPatchY; ++y)
                s_sum[y * kPitch + threadIdx.x] = run += s_sum[y * kPitch + threadIdx.x];
        }
        __syncthreads();
        const size_t base = ((size_t)p * most + k0) * kPatchTiles;
        for (uint32_t q = threadIdx.x; q < kPatchTiles; q += kThreads)
            counts[base + q] = (uint32_t)s_sum[q / kPatchX * kPitch + q % kPatchX];
        __syncthreads();
    }
}

// counts[patch][task][tile] -> entries of the tile in the patch's earlier tasks;
// totals[tile].  Eight threads share a tile's tasks: each sums its part, then
// writes the running sums.
constexpr uint32_t kRowTiles = 32, kRowParts = 8;
__global__ __launch_bounds__(kRowTiles *kRowParts) void bins_rows_kernel(uint32_t tw, uint32_t rows, uint32_t px,
                                                                       uint32_t most,
                                                                       const uint32_t *__restrict__ tasks,
                                                                       uint32_t *__restrict__ counts,
                                                                       uint32_t *__restrict__ totals) {
    constexpr uint32_t U = 16;  // rows in flight
    constexpr uint32_t kPer = kPatchTiles / kRowTiles;
    __shared__ uint32_t s_part[kRowParts][kRowTiles];
    const uint32_t i = threadIdx.x % kRowTiles, part = threadIdx.x / kRowTiles;
    const uint32_t p = blockIdx.x / kPer, tile = blockIdx.x % kPer * kRowTiles + i;
    const uint32_t n = tasks[p], per = (n + kRowParts - 1) / kRowParts;
    const uint32_t r0 = min(part * per, n), r1 = min(r0 + per, n);  // this thread's tasks
    uint32_t *const c = counts + (size_t)p * most * kPatchTiles + tile;
    uint32_t sum = 0;
    for (uint32_t r = r0; r < r1; r += U) {
        uint32_t v[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) v[u] = r + u < r1 ? c[(size_t)(r + u) * kPatchTiles] : 0u;
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) sum += v[u];
    }
    s_part[part][i] = sum;
    __syncthreads();
    uint32_t run = 0, all = 0;
#pragma unroll
    for (uint32_t q = 0; q < kRowParts; ++q) {
        run += q < part ? s_part[q][i] : 0u;
        all += s_part[q][i];
    }
    for (uint32_t r = r0; r < r1; r += U) {
        uint32_t v[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) v[u] = r + u < r1 ? c[(size_t)(r + u) * kPatchTiles] : 0u;
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            if (r + u < r1) c[(size_t)(r + u) * kPatchTiles] = run;
            run += v[u];
        }
    }
    const uint32_t x = p % px * kPatchX + tile % kPatchX, y = p / px * kPatchY + tile / kPatchX;
    if (part == 0 && x < tw && y < rows) totals[(size_t)y * tw + x] = all;
}

// offsets[tile] = entries of the tiles before it.  One workgroup.
constexpr uint32_t kOffThreads = 1024, kOffPer = 8;
__global__ __launch_bounds__(kOffThreads) void bins_offsets_kernel(uint64_t bins, const uint32_t *__restrict__ totals,
                                                                  int32_t *__restrict__ offsets) {
    __shared__ uint32_t s_wave[kOffThreads / 64];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t carry = 0;
    for (uint64_t t0 = 0; t0 < bins; t0 += kOffThreads * kOffPer) {
        const uint64_t t = t0 + (uint64_t)threadIdx.x * kOffPer;
        uint32_t v[kOffPer], n = 0;
#pragma unroll
        for (uint32_t u = 0; u < kOffPer; ++u) {
            v[u] = t + u < bins ? totals[t + u] : 0u;
            n += v[u];
        }
        uint32_t inc = n;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t w = __shfl_up(inc, o, 64);
            if ((int)lane >= o) inc += w;
        }
        if (lane == 63) s_wave[wave] = inc;
        __syncthreads();
        uint32_t run = carry + inc - n;
        for (uint32_t q = 0; q < kOffThreads / 64; ++q) {
            const uint32_t w = s_wave[q];
            run += q < wave ? w : 0u;
            carry += w;
        }
        __syncthreads();
#pragma unroll
        for (uint32_t u = 0; u < kOffPer; ++u) {
            if (t + u < bins) offsets[t + u] = (int32_t)run;
            run += v[u];
        }
    }
}

// In rows of 16 lanes: the sum of the lower lanes and the lane itself, and of all.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_or_zero(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
}
__device__ __forceinline__ uint32_t row_inclusive(uint32_t v) {
    v += dpp_or_zero<0x111>(v);  // row_shr:1
    v += dpp_or_zero<0x112>(v);
    v += dpp_or_zero<0x114>(v);
    v += dpp_or_zero<0x118>(v);
    return v;
}
__device__ __forceinline__ uint32_t row_total(uint32_t v) {
    v += dpp_or_zero<0x128>(v);  // row_ror:8
    v += dpp_or_zero<0x124>(v);
    v += dpp_or_zero<0x122>(v);
    v += dpp_or_zero<0x121>(v);
    return v;
}

__global__ __launch_bounds__(kPlaceThreads) void bins_place_kernel(
    uint32_t tw, uint32_t th, uint32_t rows, uint32_t px, uint32_t patches, uint32_t groups,
    uint32_t most, uint32_t tile_bits, const uint32_t *__restrict__ cuts, const uint32_t *__restrict__ tasks,
    const uint4 *__restrict__ records, const uint64_t *__restrict__ bits,
    const uint32_t *__restrict__ counts, const int32_t *__restrict__ offsets, int64_t *__restrict__ isect_ids,
    int32_t *__restrict__ flatten_ids, uint32_t cap) {
    constexpr uint32_t kWaves = kPlaceThreads / 64, kTiles = 64 / kTileLanes;  // tiles of a wave at a time
    __shared__ __align__(16) uint64_t s_col[kPatchX][kTileLanes];  // bit i of the 1024: pair i of the window
    __shared__ __align__(16) uint64_t s_row[kPatchY][kTileLanes];
    __shared__ uint32_t s_pos[kPatchTiles];                        // next place of each tile
    __shared__ uint32_t s_hi[kPatchY];                             // upper half of the ids of a row's first tile
    __shared__ uint2 s_pair[kWindow];                              // depth bits, flat id
    __shared__ uint32_t s_list[kWindow];
    __shared__ uint16_t s_stage[kWaves * kTiles][kStage];          // a tile's pairs, in order
    __shared__ uint32_t s_first[kMaxPatches];
    __shared__ uint32_t s_wave[kWaves];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l = lane % kTileLanes, q4 = lane / kTileLanes;
    uint16_t *const stage = s_stage[wave * kTiles + q4];
    Tasks<kPlaceThreads> all;
    all.load(tasks, patches, s_first, s_wave);
    for (uint32_t task = blockIdx.x; task < all.total; task += gridDim.x) {
        const uint32_t p = all.patch(task, s_first), k0 = task - s_first[p];
        const uint32_t *const cut = cuts + (size_t)p * (most + 1) + k0;
        const uint32_t bx = p % px * kPatchX, by = p / px * kPatchY;
        const uint32_t ph = min(kPatchY, rows - by);
        TaskBits<kPlaceThreads> sb;
        sb.load(bits + (size_t)p * groups, cut[0] * kPairGroups, cut[1] * kPairGroups, s_wave);
        const size_t base = ((size_t)p * most + k0) * kPatchTiles;
        for (uint32_t q = threadIdx.x; q < kPatchTiles; q += kPlaceThreads) {
            const uint32_t x = bx + q % kPatchX, y = by + q / kPatchX;
            const uint64_t t = (uint64_t)y * tw + x;
            s_pos[q] = x < tw && y < rows ? (uint32_t)offsets[t] + counts[base + q] : 0u;
        }
        if (threadIdx.x < kPatchY) {
            const uint32_t y = by + threadIdx.x, cam = y / th;
            s_hi[threadIdx.x] = (cam << tile_bits) | ((y - cam * th) * tw + bx);  // (the sum stays below the camera's bits)
        }
        for (uint32_t lo = 0; lo < sb.total; lo += kWindow) {
            __syncthreads();
            for (uint32_t q = threadIdx.x; q < kPatchX * kTileLanes; q += kPlaceThreads) (&s_col[0][0])[q] = 0ull;
            for (uint32_t q = threadIdx.x; q < kPatchY * kTileLanes; q += kPlaceThreads) (&s_row[0][0])[q] = 0ull;
            sb.window(lo, s_list);
            __syncthreads();
            const uint32_t n = min(kWindow, sb.total - lo);
            for (uint32_t i = threadIdx.x; i < n; i += kPlaceThreads) {
                const uint4 r = records[s_list[i]];
                s_pair[i] = make_uint2(r.y, r.x);
                const PatchBox q(r.z, r.w, bx, by);
                const uint32_t word = i >> 5, bit = 1u << (i & 31);
                for (uint32_t x = q.x0; x < q.x1; ++x) atomicOr(reinterpret_cast<uint32_t *>(s_col[x]) + word, bit);
                for (uint32_t y = q.y0; y < q.y1; ++y) atomicOr(reinterpret_cast<uint32_t *>(s_row[y]) + word, bit);
            }
            __syncthreads();
            constexpr uint32_t kSteps = kPatchX / kTiles;  // steps of a row
            for (uint32_t it = wave; it < ph * kSteps; it += kWaves) {
                // (skewed: each wave meets every column, also where the pairs crowd a few)
                const uint32_t y = it / kSteps, x = (it + y) % kSteps * kTiles + q4;
                uint64_t m = s_col[x][l] & s_row[y][l];
                if (__ballot(m != 0ull) == 0ull) continue;
                const uint32_t c = (uint32_t)__popcll(m), cnt = row_total(c);
                uint32_t at = row_inclusive(c) - c;
                const uint32_t pos = s_pos[y * kPatchX + x];
                const uint64_t hi = (uint64_t)(s_hi[y] + x) << 32;
                for (uint32_t s0 = 0;; s0 += kStage) {
                    while (m && at < s0 + kStage) {
                        stage[at - s0] = (uint16_t)(l * 64 + (uint32_t)__builtin_ctzll(m));
                        m &= m - 1;
                        ++at;
                    }
                    __builtin_amdgcn_wave_barrier();  // (this wave's LDS accesses are in order)
                    const uint32_t end = min(cnt, s0 + kStage);
                    for (uint32_t k = s0 + l; k < end; k += kTileLanes) {
                        const uint2 pr = s_pair[stage[k - s0]];
                        if (pos + k < cap) {  // entries past a capacity are not stored
                            isect_ids[pos + k] = (int64_t)(hi | pr.x);
                            flatten_ids[pos + k] = (int32_t)pr.y;
                        }
                    }
                    __builtin_amdgcn_wave_barrier();
                    if (__ballot(cnt > s0 + kStage) == 0ull) break;
                }
                if (l == 0) s_pos[y * kPatchX + x] = pos + cnt;
            }
        }
        __syncthreads();
    }
}

}  // namespace ubs

using namespace ubs;

extern "C" {

size_t ubs_isect_bins_workspace_bytes(uint32_t C, uint32_t N, uint32_t tw, uint32_t th) {
    BinShape s;
    return bin_shape(C, N, tw, th, s) ? s.bytes : 0;
}

int ubs_isect_bins_pays(uint32_t C, uint32_t N, uint32_t tw, uint32_t th, int64_t n_isects) {
    BinShape s;
    return bin_shape(C, N, tw, th, s) ? bins_pays((uint64_t)C * N, s.bins, s.patches, n_isects) : 0;
}

static int bins_check(uint32_t C, uint32_t N, uint32_t tw, uint32_t th, const void *ws, size_t ws_bytes, BinShape &s) {
    UBS_REQUIRE(bin_shape(C, N, tw, th, s), "tile grid or pair count past the direct placement's limits");
    UBS_REQUIRE(bit_width_u32(tw * th) + bit_width_u32(C) <= 32, "camera and tile ids need more than 32 bits");
    if (!ws || ws_bytes < s.bytes) {
        set_error("isect workspace too small (%zu < %zu)", ws_bytes, s.bytes);
        return UBS_ERR_WORKSPACE;
    }
    return UBS_OK;
}

int ubs_isect_bins_plan(uint32_t C, uint32_t N, const void *pair_records, const int32_t *order, uint32_t ts,
                        uint32_t tw, uint32_t th, int32_t *tile_offsets, void *workspace, size_t ws_bytes,
                        void *stream) {
    BinShape s;
    UBS_REQUIRE(ts > 0, "tile_size must be > 0");
    UBS_REQUIRE(pair_records && order && tile_offsets, "null pointer");
    const int rc = bins_check(C, N, tw, th, workspace, ws_bytes, s);
    if (rc != UBS_OK) return rc;
    hipStream_t st = as_stream(stream);
    char *ws = static_cast<char *>(workspace);
    uint4 *records = reinterpret_cast<uint4 *>(ws);
    uint64_t *bits = reinterpret_cast<uint64_t *>(ws + s.bits);
    uint32_t *cuts = reinterpret_cast<uint32_t *>(ws + s.cuts), *tasks = reinterpret_cast<uint32_t *>(ws + s.tasks);
    uint32_t *sums = reinterpret_cast<uint32_t *>(ws + s.sums);
    uint32_t *counts = reinterpret_cast<uint32_t *>(ws + s.counts), *totals = reinterpret_cast<uint32_t *>(ws + s.totals);
    bins_pairs_kernel<<<s.groups / kPairGroups, kThreads, 0, st>>>((uint32_t)((uint64_t)C * N), N,
                                                                  static_cast<const float4 *>(pair_records), order, ts,
                                                                  tw, th, s.px, s.patches, s.groups, records, bits, sums);
    UBS_LAUNCH_CHECK("bins_pairs_kernel");
    bins_cuts_kernel<<<s.patches, kCutThreads, 0, st>>>(s.groups / kPairGroups, s.most, sums, cuts, tasks);
    UBS_LAUNCH_CHECK("bins_cuts_kernel");
    const uint32_t blocks = (uint32_t)std::min((uint64_t)s.patches * s.most, (uint64_t)kCountBlocks);
    bins_count_kernel<<<blocks, kThreads, 0, st>>>(tw, C * th, s.px, s.patches, s.groups, s.most, cuts, tasks, records,
                                                 bits, counts);
    UBS_LAUNCH_CHECK("bins_count_kernel");
    bins_rows_kernel<<<s.patches * (kPatchTiles / kRowTiles), kRowTiles * kRowParts, 0, st>>>(tw, C * th, s.px, s.most,
                                                                                            tasks, counts, totals);
    UBS_LAUNCH_CHECK("bins_rows_kernel");
    bins_offsets_kernel<<<1, kOffThreads, 0, st>>>(s.bins, totals, tile_offsets);
    UBS_LAUNCH_CHECK("bins_offsets_kernel");
    return UBS_OK;
}

int ubs_isect_bins_place(uint32_t C, uint32_t N, uint32_t tw, uint32_t th, const int32_t *tile_offsets,
                         const void *workspace, size_t ws_bytes, int64_t *isect_ids, int32_t *flatten_ids,
                         int64_t n_isects, void *stream) {
    BinShape s;
    UBS_REQUIRE(n_isects >= 0 && n_isects < (1ll << 31), "n_isects must be in [0, 2^31)");
    const int rc = bins_check(C, N, tw, th, workspace, ws_bytes, s);
    if (rc != UBS_OK) return rc;
    if (n_isects == 0) return UBS_OK;
    UBS_REQUIRE(tile_offsets && isect_ids && flatten_ids, "null pointer");
    const char *ws = static_cast<const char *>(workspace);
    const uint32_t blocks = (uint32_t)std::min((uint64_t)s.patches * s.most, (uint64_t)kPlaceBlocks);
    bins_place_kernel<<<blocks, kPlaceThreads, 0, as_stream(stream)>>>(
        tw, th, C * th, s.px, s.patches, s.groups, s.most, bit_width_u32(tw * th),
        reinterpret_cast<const uint32_t *>(ws + s.cuts), reinterpret_cast<const uint32_t *>(ws + s.tasks),
        reinterpret_cast<const uint4 *>(ws), reinterpret_cast<const uint64_t *>(ws + s.bits),
        reinterpret_cast<const uint32_t *>(ws + s.counts), tile_offsets, isect_ids, flatten_ids, (uint32_t)n_isects);
    UBS_LAUNCH_CHECK("bins_place_kernel");
    return UBS_OK;
}

}  // extern "C"
