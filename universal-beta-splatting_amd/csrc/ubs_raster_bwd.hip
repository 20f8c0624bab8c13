// Backward tile blend of Beta primitives on gfx950.
//
// One wave per 8x8 sub-block of a tile, its own workgroup: the waves share
// nothing and never wait for each other.  A wave walks its tile's list back to
// front from its largest last contributor, 64 entries at a time; entries whose
// support reaches the sub-block (the mask the forward kept, or the forward's
// test again) are queued in LDS, and the queue is blended in groups of up to 32
// primitives with the primitives across the lanes: lane l holds primitives
// 2 (l & 15) and 2 (l & 15) + 1 of the group and, in step b, the pixels
// 8 b + 2 (l >> 4) + {0, 1} of the sub-block, so that a row of 16 lanes has one
// pixel and 32 primitives, back to front.
//   * A pixel's transmittance before each primitive is the state left by the
//     groups behind it times the inclusive product over the row of
//     1 / (1 - alpha), and the colour behind it the exclusive sum of
//     alpha T (c . v): two 16-lane scans of four DPP steps each.  The
//     recovery starts from the exact T after the last contributor (kept by the
//     forward) and divides by this kernel's 1 - alpha.  sigma has the forward's
//     bits; alpha = o (1 - sigma)^(beta - 1) (1 - sigma) here and
//     o (1 - sigma)^beta there agree to about (3 + beta |log2(1 - sigma)|) 2^-23
//     relative, and each primitive passed moves T by that times
//     alpha / (1 - alpha).
//   * A primitive's gradients (rasterize_to_pixels_bwd.cu:200-247) add up in
//     its own lane's registers over the steps; the four rows are summed once
//     per group (two permlane levels), turned through LDS so that 16
//     consecutive lanes hold one primitive's record, and added to global
//     memory with hardware float atomics, one 64-byte line per (sub-block,
//     primitive).
//   * The pixels share work: a lane's pixels have one of two x offsets (kept
//     for the whole group) and a step one y offset, and the gradient's moments
//     are formed from sums of v_sigma and dy v_sigma per x offset.
//   * More than 4 channels: one primitive per lane and four pixels per step,
//     with the contractions on the matrix cores, which hold the same layout
//     (c . v of 16 primitives x 16 pixels is one v_mfma_f32_16x16x4_f32 per 4
//     channels, the colour gradient sum alpha T v one per pixel and 16
//     channels, FP32 throughout).
//
// Why: with a pixel per lane (the layout before) every (wave, primitive) step
// summed 10 values over the 64 lanes and added them to LDS accumulators: of
// 311 SIMD cycles a step ~108 were cross-lane reduction, and ds_add_f32 takes
// ~3 LDS cycles for every active lane (64 lanes: 193; ds_add_u32: 4.7), ~120
// more.  Here a primitive costs no reduction, 4.5 DPP operations per evaluation
// and no LDS atomic.  Blocks of four waves over a shared staged batch took 1.70
// ms where this takes 1.46: a barrier per batch, a tenth of the group slots
// empty.  What bounds it now: VALU issue (~40 instructions per evaluation; an
// FP32 multiply-add pairs with another wave's at ~2.4 cycles, a DPP operation
// takes ~4, a log2 / exp2 / reciprocal ~8), then the line rate of the atomics
// (20 G/s: 0.9 ms of it under the blend at 18M lines).  1080p, 1M primitives
// (23M evaluations of 64): 2.71 -> 1.49 ms; 8 views of 3M: 24.8 -> 14.3 ms.
// The T recovery can run in fp64 (template flag) where stability needs it.
#pragma clang fp contract(off)

#include <type_traits>

#include "ubs_raster.h"

namespace ubs {

// Waves per SIMD the registers are held to (LDS would allow five).
#ifndef UBS_BWD_WAVES_PER_EU
#define UBS_BWD_WAVES_PER_EU 4
#endif
// Primitives per lane in a full group: two consecutive ones share each scan
// (4.5 DPP operations per evaluation instead of 9) and the reads of the pixel
// state; three waves' worth of registers more.
#ifndef UBS_BWD_PRIMS
#define UBS_BWD_PRIMS 2
#endif

// A wave's priority is raised through its bursts of transcendental and DPP
// operations.  The SIMD pairs FP32 operations of two waves only while no such
// operation of a third comes in between; issued in a burst they leave the
// others' runs of plain operations whole.  The instruction mix of the blend
// loop takes 2.65 instead of 4.05 cycles per instruction with it, this kernel
// 2.29 instead of 2.49 ms (before its other changes).
#define UBS_PRIO_ON "s_setprio 3\n\t"
#define UBS_PRIO_OFF "s_setprio 0\n\t"

// Inclusive scans over the 16 lanes of every row, two or four registers at a
// time (a DPP read of a register needs two wait states after its write: the
// other registers' instructions, and the s_nops).  row_shr:N leaves the lanes
// below N as they are; with bound_ctrl:0 they read zeros.
#define UBS_DPP(OP, D, S, SHR, BC) OP " " D ", " S ", " S " row_shr:" SHR " row_mask:0xf bank_mask:0xf" BC "\n\t"
#define UBS_SCAN2(OP, SHR) "s_nop 0\n\t" UBS_DPP(OP, "%0", "%0", SHR, "") UBS_DPP(OP, "%1", "%1", SHR, "")
#define UBS_SCAN4(OP, SHR)                                                                  \
    UBS_DPP(OP, "%0", "%0", SHR, "") UBS_DPP(OP, "%1", "%1", SHR, "")                       \
    UBS_DPP(OP, "%2", "%2", SHR, "") UBS_DPP(OP, "%3", "%3", SHR, "")
__device__ __forceinline__ void row_scan_mul(float (&x)[2]) {
    asm(UBS_PRIO_ON "s_nop 0\n\t" UBS_SCAN2("v_mul_f32_dpp", "1") UBS_SCAN2("v_mul_f32_dpp", "2")
            UBS_SCAN2("v_mul_f32_dpp", "4") UBS_SCAN2("v_mul_f32_dpp", "8") UBS_PRIO_OFF
        : "+v"(x[0]), "+v"(x[1]));
}
__device__ __forceinline__ void row_scan_mul(float (&x)[4]) {
    asm(UBS_PRIO_ON "s_nop 1\n\t" UBS_SCAN4("v_mul_f32_dpp", "1") UBS_SCAN4("v_mul_f32_dpp", "2")
            UBS_SCAN4("v_mul_f32_dpp", "4") UBS_SCAN4("v_mul_f32_dpp", "8") UBS_PRIO_OFF
        : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]));
}
__device__ __forceinline__ void row_scan_add(const float (&x)[2], float (&o)[2]) {
    asm(UBS_PRIO_ON "s_nop 1\n\t" UBS_DPP("v_add_f32_dpp", "%0", "%2", "1", " bound_ctrl:0")
            UBS_DPP("v_add_f32_dpp", "%1", "%3", "1", " bound_ctrl:0") UBS_SCAN2("v_add_f32_dpp", "2")
                UBS_SCAN2("v_add_f32_dpp", "4") UBS_SCAN2("v_add_f32_dpp", "8") UBS_PRIO_OFF
        : "=&v"(o[0]), "=&v"(o[1])
        : "v"(x[0]), "v"(x[1]));
}
__device__ __forceinline__ void row_scan_add(const float (&x)[4], float (&o)[4]) {
    asm(UBS_PRIO_ON "s_nop 1\n\t" UBS_DPP("v_add_f32_dpp", "%0", "%4", "1", " bound_ctrl:0")
            UBS_DPP("v_add_f32_dpp", "%1", "%5", "1", " bound_ctrl:0")
                UBS_DPP("v_add_f32_dpp", "%2", "%6", "1", " bound_ctrl:0")
                    UBS_DPP("v_add_f32_dpp", "%3", "%7", "1", " bound_ctrl:0") UBS_SCAN4("v_add_f32_dpp", "2")
                        UBS_SCAN4("v_add_f32_dpp", "4") UBS_SCAN4("v_add_f32_dpp", "8") UBS_PRIO_OFF
        : "=&v"(o[0]), "=&v"(o[1]), "=&v"(o[2]), "=&v"(o[3])
        : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]));
}
#undef UBS_SCAN4
#undef UBS_SCAN2
#undef UBS_DPP
#undef UBS_PRIO_ON
#undef UBS_PRIO_OFF

// value of lane l - N of the row, 1 in the lanes below N
template <int N>
__device__ __forceinline__ double row_shr_or_one(double x) {
    const double one = 1.0;
    const int2 v = __builtin_bit_cast(int2, x), o = __builtin_bit_cast(int2, one);
    int2 r;
    r.x = __builtin_amdgcn_update_dpp(o.x, v.x, 0x110 + N, 0xf, 0xf, false);
    r.y = __builtin_amdgcn_update_dpp(o.y, v.y, 0x110 + N, 0xf, 0xf, false);
    return __builtin_bit_cast(double, r);
}
// value of lane l - 1 of the row, 0 in lane 0
__device__ __forceinline__ float row_shr1_or_zero(float x) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(x), 0x111, 0xf, 0xf, true));
}

template <int R>
__device__ __forceinline__ void row_scan_mul(double (&x)[R]) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
        x[r] *= row_shr_or_one<1>(x[r]);
        x[r] *= row_shr_or_one<2>(x[r]);
        x[r] *= row_shr_or_one<4>(x[r]);
        x[r] *= row_shr_or_one<8>(x[r]);
    }
}

// LDS written and read by one wave only: its LDS operations complete in
// order, so it is enough that the compiler keeps them in order.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// STATS (measurement builds only; the library's kernels have it off) counts
// into stats[0..6]: (wave, primitive) evaluations, lane evaluations at or
// before the pixel's last contributor, of those that contribute, groups of 16
// primitives, staged entries, groups on the fast path, and empty primitive
// slots in the groups.
template <int TS, int CDIM, bool F64T, bool STATS = false>
__global__ __launch_bounds__(64, UBS_BWD_WAVES_PER_EU) void raster_bwd_kernel(
    uint32_t C, uint32_t N, int64_t n_isects, uint32_t channels, uint32_t coff,
    const float *__restrict__ means2d, const float *__restrict__ conics, const float *__restrict__ colors,
    const float *__restrict__ opacities, const float *__restrict__ betas, const float *__restrict__ backgrounds,
    const uint8_t *__restrict__ masks, uint32_t W, uint32_t H, uint32_t tw, uint32_t th,
    const int32_t *__restrict__ tile_offsets, const int32_t *__restrict__ flatten_ids,
    const float *__restrict__ render_alphas, const int32_t *__restrict__ last_ids, const float *__restrict__ T_final,
    const float *__restrict__ v_render_colors, const float *__restrict__ v_render_alphas,
    float *__restrict__ v_means2d, float *__restrict__ v_conics, float *__restrict__ v_colors,
    float *__restrict__ v_opacities, float *__restrict__ v_betas, const float4 *__restrict__ rec, int wide_rec,
    float *__restrict__ vrec, const float *__restrict__ T_ckpt, unsigned long long *__restrict__ stats = nullptr,
    const uint32_t *__restrict__ order = nullptr, unsigned long long *__restrict__ wg_times = nullptr,
    const void *__restrict__ entry_masks = nullptr) {
    constexpr int SB = TS / 8;               // sub-blocks per tile side
    constexpr int BS = TS * TS;              // entries per checkpointed batch
    constexpr int NCOL = CDIM <= 4 ? 4 : CDIM;
    constexpr bool kMfma = CDIM > 4;         // the channel contractions on the matrix cores (their depth: 4 channels)
    constexpr int NCD = NCOL / 4;            // MFMAs of one c . v
    constexpr int NFD = (CDIM + 15) / 16;    // 16-channel blocks of the colour gradient
    constexpr int R = kMfma ? 4 : 2;         // pixels per lane and step
    constexpr int STEPS = 16 / R;
    constexpr int MMAX = kMfma ? 1 : UBS_BWD_PRIMS;  // primitives per lane
    constexpr int QN = 64 + 16 * MMAX;       // queue slots: a chunk on top of less than a group
    constexpr int kTrStride = 13;            // 12 values, and odd: 16 primitives hit different banks
    constexpr uint32_t kPlainBit = 1u << 31;  // of a queued isect index
    using TT = typename std::conditional<F64T, double, float>::type;
    typedef float f4 __attribute__((ext_vector_type(4)));
    // the sub-block's queued primitives, back to front, as a ring
    __shared__ float4 q_geo[QN];    // x, y, a, 2b
    __shared__ float4 q_geo2[QN];   // c, opacity, beta, id (bits)
    __shared__ float4 q_colv[kMfma ? 1 : QN];
    __shared__ float q_col[kMfma ? CDIM : 1][kMfma ? QN : 1];
    constexpr bool kIdxInCol = CDIM <= 3;  // isect index | kPlainBit: the colour's free word, or its own
    __shared__ uint32_t q_idx[kIdxInCol ? 1 : QN];
    // the state of the 64 pixels: T behind the primitives still to come, the
    // rest of d/d(alpha) (T_final (v_alpha_out - bg . v) - colour behind . v),
    // the colour gradient (rows of channels; for the MFMA the pixel index is
    // xored with 16 (channel & 3) so that its reads of four channels hit
    // different banks) and the last contributor
    struct __align__(16) Pixels {
        TT T[64];
        float P[64];
        float v[CDIM][64];
        int32_t bin[64];
    };
    __shared__ Pixels px;
    __shared__ float s_tr[16 * kTrStride + 4];  // a group's totals, [primitive][value], on their way to memory

    // workgroup -> (tile, sub-block): the sub-blocks of a tile are consecutive
    // workgroups of one XCD, and share its L2's copy of the tile's records
    constexpr uint32_t NSUB = SB * SB;
    uint32_t logical;
    const uint32_t slot = blockIdx.x / kNumXcd;
    if (!xcd_tile(blockIdx.x % kNumXcd + kNumXcd * (slot / NSUB), C, tw, th, logical, order)) return;
    const uint32_t sub = slot % NSUB;
    // (measurement builds: the workgroup's start on the constant-rate clock)
    unsigned long long t_start = 0;
    if constexpr (STATS) t_start = __builtin_amdgcn_s_memrealtime();
    const uint32_t cam = logical / (th * tw);
    const uint32_t tile = logical % (th * tw);
    const uint32_t ty = tile / tw, tx = tile % tw;
    if (masks && !masks[(size_t)cam * th * tw + tile]) return;

    const int lane = threadIdx.x;
    const int li = lane & 15, row = lane >> 4;
    const uint32_t sx0 = tx * TS + (sub % SB) * 8, sy0 = ty * TS + (sub / SB) * 8;  // the sub-block's first pixel
    const uint32_t i = sy0 + (lane >> 3), j = sx0 + (lane & 7);
    const bool inside = i < H && j < W;
    const int64_t pix = (int64_t)cam * H * W + (int64_t)i * W + j;
    const bool first_chunk = (coff == 0);

    const int64_t tbase = (int64_t)cam * th * tw;
    // a valid sort gives ordered offsets within [0, n_isects]; the clamps keep
    // the lists of a sort that gave up on a look-back wait inside the buffers
    const int32_t off_hi = (cam == C - 1 && tile == th * tw - 1) ? (int32_t)n_isects : tile_offsets[tbase + tile + 1];
    const int32_t range_start = min(max(tile_offsets[tbase + tile], 0), (int32_t)n_isects);
    const int32_t range_end = min(max(off_hi, range_start), (int32_t)n_isects);

    // ---- per-pixel state: thread -> pixel `lane` of the sub-block.  Pixels
    // outside the image get T = 0, zero gradients and no last contributor: no
    // primitive is valid there.
    const int32_t bin_final = inside ? last_ids[pix] : 0;
    bool finite = true;  // no infinity or NaN in the incoming gradients
    {
        const float Tf = inside ? (T_final ? T_final[pix] : 1.f - render_alphas[pix]) : 0.f;
        float bg_dot = 0.f;
#pragma unroll
        for (int k = 0; k < CDIM; ++k) {
            const float v = inside ? v_render_colors[pix * channels + coff + k] : 0.f;
            if (backgrounds) bg_dot = __builtin_fmaf(backgrounds[cam * channels + coff + k], v, bg_dot);
            finite = finite && fabsf(v) < __builtin_huge_valf();
            px.v[k][kMfma ? lane ^ (16 * (k & 3)) : lane] = v;
        }
        const float vra = (inside && first_chunk && v_render_alphas) ? v_render_alphas[pix] : 0.f;  // null: zeros
        px.T[lane] = (TT)Tf;
        const float P = Tf * (vra - bg_dot);  // vra - bg_dot: d/d(T_final) of the pixel's outputs
        finite = finite && fabsf(P) < __builtin_huge_valf();
        px.P[lane] = P;
        px.bin[lane] = inside ? bin_final : INT32_MIN;
    }
    const bool all_finite = __ballot(finite) == ~0ull;
    // the largest last contributor over the wave bounds the useful range; up
    // to the smallest, every pixel is still blending.  A pixel outside the image
    // never is (nothing stopped at T <= 1e-4 there, so the product of 1 / (1 -
    // alpha) over a stack of opaque primitives would pass FP32's range, and 0 x
    // inf is NaN): a sub-block over the image's edge takes the general tests.
    const int32_t wave_bin_max = __builtin_amdgcn_readfirstlane(wave_max_i32(bin_final));
    const int32_t wave_bin_min = -__builtin_amdgcn_readfirstlane(wave_max_i32(inside ? -bin_final : INT32_MAX));
    // the lane's pixels: x offsets pxb + r, y offset pyb + the step's
    const float pxb = (float)(sx0 + (uint32_t)(R == 4 ? 4 * (row & 1) : 2 * row)) + 0.5f;
    const float pyb = (float)(sy0 + (uint32_t)(R == 4 ? row >> 1 : 0)) + 0.5f;

    // Where the lane's value of a primitive's gradient goes (lane li of a row:
    // value li of xy, conic, opacity, beta; from lane 8 the colours of up to 4
    // channels): grad_base + id * grad_stride.
    const bool grad_lane = li < 7 || (!kMfma && li >= 8 && li < 8 + CDIM);
    float *grad_base;
    int grad_stride;
    if (li >= 8 && !(vrec && wide_rec)) {
        grad_base = v_colors + coff + (li - 8);
        grad_stride = (int)channels;
    } else if (vrec) {
        grad_base = vrec + li;
        grad_stride = wide_rec ? (int)kWideRecordFloats : (int)kRecordFloats;
    } else {
        grad_base = li < 2 ? v_means2d + li : li < 5 ? v_conics + (li - 2) : li == 5 ? v_opacities : v_betas;
        grad_stride = li < 2 ? 2 : li < 5 ? 3 : 1;
    }

    uint32_t st_steps = 0, st_live = 0, st_valid = 0, st_groups = 0, st_staged = 0, st_fast = 0, st_empty = 0;
    int q_head = 0, q_count = 0;  // wave-uniform
    // The group at the queue's head: up to 16 M primitives, M per lane.
    auto group = [&](auto m_tag) {
        constexpr int M = decltype(m_tag)::value;  // primitives per lane, back to front
        bool has[M];
        uint32_t idx[M];
        float4 g1[M], g2[M];
        float cl[M][kMfma ? NCD : CDIM];  // the colour; for the MFMA, the row's channel of every block of four
        bool plain = true;
        const int left = q_count;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            has[m] = M * li + m < left;
            int e = q_head + (has[m] ? M * li + m : 0);
            e = e >= QN ? e - QN : e;
            idx[m] = kIdxInCol ? __float_as_uint(q_colv[kMfma ? 0 : e].w) : q_idx[kIdxInCol ? 0 : e];
            plain = plain && (idx[m] & kPlainBit);
            idx[m] &= ~kPlainBit;
            g1[m] = q_geo[e];
            g2[m] = q_geo2[e];
#pragma unroll
            for (int c = 0; c < (kMfma ? NCD : CDIM); ++c)
                cl[m][c] = kMfma ? q_col[kMfma ? 4 * c + row : 0][kMfma ? e : 0]
                                 : reinterpret_cast<const float *>(&q_colv[kMfma ? 0 : e])[c];
            if (!has[m]) g1[m].x = __builtin_huge_valf();  // sigma is infinite or NaN: contributes nowhere
        }
        // A group whose entries all precede every pixel's last contributor
        // and whose primitives are plain leaves out the tests that cannot fail.
        const int32_t first_idx = (int32_t)__builtin_amdgcn_readfirstlane(idx[0]);  // the group's largest
        const bool fast = all_finite && first_idx <= wave_bin_min && __ballot(plain) == ~0ull;
        if constexpr (STATS) {
            const uint32_t k = (uint32_t)min(left, 16 * M);
            st_steps += k;
            st_groups += 1;
            st_empty += 16u * M - k;
            st_fast += (uint32_t)fast;
        }
        float dx[M][R], adx[M][R], bdx[M][R], bm1[M];
        // sums over the lane's 16 pixels (va: the gradient of alpha, sg = va
        // (1 - sigma)^(beta - 1)): per x offset of sg and dy sg, and of
        // dy^2 sg, va (1 - sigma)^beta, the latter x log2(1 - sigma), and
        // per channel of alpha T v
        float sA[M][R], sB[M][R], sum[M][3], scol[M][kMfma ? 1 : CDIM];
#pragma unroll
        for (int m = 0; m < M; ++m) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                dx[m][r] = g1[m].x - (pxb + (float)r);
                adx[m][r] = g1[m].z * dx[m][r];
                bdx[m][r] = g1[m].w * dx[m][r];
                sA[m][r] = sB[m][r] = 0.f;
            }
            bm1[m] = g2[m].z - 1.f;
            sum[m][0] = sum[m][1] = sum[m][2] = 0.f;
#pragma unroll
            for (int k = 0; k < (kMfma ? 1 : CDIM); ++k) scol[m][k] = 0.f;
        }
        f4 dcol[NFD];  // the channel sums from the MFMA, [primitive][channel]
#pragma unroll
        for (int s = 0; s < NFD; ++s) dcol[s] = (f4){0.f, 0.f, 0.f, 0.f};
        auto steps = [&](auto fast_tag) {
            constexpr bool FAST = decltype(fast_tag)::value;
            struct Pix {  // a step's pixels (state read from LDS one step ahead)
                TT T[R];
                float P[R], v[kMfma ? 1 : CDIM][R];
                int32_t bin[R];
            };
            auto load_r = [&](const auto *src, auto (&dst)[R]) {
                if constexpr (R == 4 && sizeof(dst[0]) == 4) {
                    const float4 q = *reinterpret_cast<const float4 *>(src);
                    __builtin_memcpy(dst, &q, sizeof(q));
                } else if constexpr (R == 2 && sizeof(dst[0]) == 4) {
                    const float2 q = *reinterpret_cast<const float2 *>(src);
                    __builtin_memcpy(dst, &q, sizeof(q));
                } else {
#pragma unroll
                    for (int r = 0; r < R; ++r) dst[r] = src[r];
                }
            };
            auto load_pix = [&](const int p, Pix &x) {
                if constexpr (!kMfma) {
#pragma unroll
                    for (int k = 0; k < CDIM; ++k) load_r(&px.v[k][p], x.v[k]);
                }
                load_r(&px.T[p], x.T);
                load_r(&px.P[p], x.P);
                if constexpr (!FAST || STATS) load_r(&px.bin[p], x.bin);
            };
            float py = pyb;
            int p0 = R * row;  // the row's R pixels of the step
#pragma unroll 1
            for (int pb = 0; pb < STEPS; ++pb, p0 += 4 * R, py += (float)(R / 2)) {
                Pix cur;
                load_pix(p0, cur);
                TT(&T0)[R] = cur.T;
                float(&P0)[R] = cur.P;
                auto &vv = cur.v;
                int32_t(&bin)[R] = cur.bin;
                float cd[M][R];  // c . v of the lane's primitives with its pixels
                if constexpr (kMfma) {
                    f4 acc = (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int c = 0; c < NCD; ++c)
                        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(
                            px.v[4 * c + row][(16 * pb + li) ^ (16 * row)], cl[0][c], acc, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < R; ++r) cd[0][r] = acc[r];
                }
                float dy[M], oms[M][R], lg[M][R], pm1[M][R], vis[M][R], ov[M][R], alpha[M][R], oma[M][R], ra[M][R];
                bool valid[M][R];
                TT rt[M][R], scan[R];
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    dy[m] = g1[m].y - py;
                    const float cyy = (g2[m].x * dy[m]) * dy[m];
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const float sigma =
                            __builtin_fmaf(bdx[m][r], dy[m], __builtin_fmaf(adx[m][r], dx[m][r], cyy));
                        if constexpr (FAST)  // 0 <= sigma < 1 (sigma is not -0 here)
                            valid[m][r] = __float_as_uint(sigma) < 0x3f800000u;
                        else
                            valid[m][r] = sigma >= 0.f && sigma < 1.f && (int32_t)idx[m] <= bin[r];
                        if constexpr (STATS) {
                            st_live += (uint32_t)(has[m] && (int32_t)idx[m] <= bin[r]);
                            st_valid += (uint32_t)valid[m][r];
                        }
                        oms[m][r] = valid[m][r] ? 1.f - sigma : 1.f;
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_setprio(3);
#pragma unroll
                for (int m = 0; m < M; ++m)
#pragma unroll
                    for (int r = 0; r < R; ++r) lg[m][r] = __builtin_amdgcn_logf(oms[m][r]);  // log2(1 - sigma)
                // (1-sigma)^(beta-1) by one exp2, (1-sigma)^beta from it by one
                // multiply (one transcendental fewer than two exp2)
#pragma unroll
                for (int m = 0; m < M; ++m)
#pragma unroll
                    for (int r = 0; r < R; ++r) pm1[m][r] = __builtin_amdgcn_exp2f(bm1[m] * lg[m][r]);
                __builtin_amdgcn_s_setprio(0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int m = 0; m < M; ++m)
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        if constexpr (FAST) pm1[m][r] = valid[m][r] ? pm1[m][r] : 0.f;
                        vis[m][r] = pm1[m][r] * oms[m][r];
                        ov[m][r] = g2[m].y * vis[m][r];
                        alpha[m][r] = FAST ? ov[m][r] : (valid[m][r] ? fminf(0.999f, ov[m][r]) : 0.f);
                        oma[m][r] = 1.f - alpha[m][r];
                        if constexpr (F64T) {
                            rt[m][r] = 1.0 / (1.0 - (double)alpha[m][r]);
                            ra[m][r] = (float)rt[m][r];
                        } else {
                            rt[m][r] = ra[m][r] = __builtin_amdgcn_rcpf(oma[m][r]);
                        }
                    }
#pragma unroll
                for (int r = 0; r < R; ++r) scan[r] = M == 2 ? rt[0][r] * rt[M - 1][r] : rt[0][r];
                row_scan_mul(scan);
                float Tc[M][R], fac[M][R], x[M][R], xl[R], xs[R], w[R];
                if constexpr (!kMfma) {
#pragma unroll
                    for (int m = 0; m < M; ++m)
#pragma unroll
                        for (int r = 0; r < R; ++r) {
                            cd[m][r] = cl[m][0] * vv[0][r];
#pragma unroll
                            for (int k = 1; k < CDIM; ++k) cd[m][r] = __builtin_fmaf(cl[m][k], vv[k][r], cd[m][r]);
                        }
                }
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    T0[r] *= scan[r];  // T before the lane's frontmost primitive
                    Tc[M - 1][r] = (float)T0[r];
                    // (the one behind it: T before it, times 1 - alpha of the front one)
                    if constexpr (M == 2)
                        Tc[0][r] = F64T ? (float)(T0[r] * (TT)(1.0 - (double)alpha[1][r])) : Tc[1][r] * oma[1][r];
#pragma unroll
                    for (int m = 0; m < M; ++m) {
                        fac[m][r] = alpha[m][r] * Tc[m][r];
                        x[m][r] = cd[m][r] * fac[m][r];
                    }
                    xl[r] = M == 2 ? x[0][r] + x[M - 1][r] : x[0][r];
                }
                row_scan_add(xl, xs);
                if constexpr (!kMfma) {
#pragma unroll
                    for (int m = 0; m < M; ++m)
#pragma unroll
                        for (int k = 0; k < CDIM; ++k)
#pragma unroll
                            for (int r = 0; r < R; ++r)
                                scol[m][k] = __builtin_fmaf(fac[m][r], vv[k][r], scol[m][k]);
                }
                float behind[M][R];  // the state behind each primitive
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    w[r] = P0[r] - xs[r];
                    behind[0][r] = P0[r] - row_shr1_or_zero(xs[r]);
                    if constexpr (M == 2) behind[1][r] = behind[0][r] - x[0][r];
                }
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    float ysum = 0.f;
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const float v_alpha = __builtin_fmaf(Tc[m][r], cd[m][r], ra[m][r] * behind[m][r]);
                        // geometry, opacity and beta get gradient only below the 0.999 clamp
                        const float va = FAST ? v_alpha : ((valid[m][r] && ov[m][r] <= 0.999f) ? v_alpha : 0.f);
                        // v_sigma = -opac beta va pm1; the per-primitive factors are applied
                        // once per (tile, primitive) at the flush
                        const float sg = va * pm1[m][r];
                        sA[m][r] += sg;
                        sB[m][r] = __builtin_fmaf(dy[m], sg, sB[m][r]);
                        ysum = r == 0 ? sg : ysum + sg;
                        const float sv = vis[m][r] * va;
                        sum[m][1] += sv;
                        sum[m][2] = __builtin_fmaf(sv, lg[m][r], sum[m][2]);
                    }
                    sum[m][0] = __builtin_fmaf(dy[m] * dy[m], ysum, sum[m][0]);
                }
                if constexpr (kMfma) {
#pragma unroll
                    for (int s = 0; s < NFD; ++s) {
                        // (8 channels: lanes past them repeat a channel, unused)
                        const int ch = 16 * s + (CDIM < 16 ? li & (CDIM - 1) : li);
                        float v4[R];
                        load_r(&px.v[ch][p0 ^ (16 * (ch & 3))], v4);
#pragma unroll
                        for (int r = 0; r < R; ++r)
                            dcol[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(fac[0][r], v4[r], dcol[s], 0, 0, 0);
                    }
                }
                if (li == 15) {  // the row's frontmost primitive leaves the pixels' state
#pragma unroll
                    for (int r = 0; r < R; ++r) px.T[p0 + r] = T0[r];
#pragma unroll
                    for (int r = 0; r < R; ++r) px.P[p0 + r] = w[r];
                }
            }
            wave_lds_fence();
        };
        if (fast)
            steps(std::true_type{});
        else
            steps(std::false_type{});
        // ---- the primitives' gradients: x moments from the sums per x
        // offset (su = sum dx sg, sw = sum dy sg, then dx^2, dx dy, dy^2),
        // the conic and the factors that are constant per primitive; then
        // the four rows are summed (two permlane levels leave row Q with
        // value 2 (Q & 1) + (Q >> 1) of four) and every lane adds its total
        // to the primitive's gradient record in global memory.
        int lane_o = lane;  // (opaque, as above)
        asm volatile("" : "+v"(lane_o));
        const int li = lane_o & 15, row = lane_o >> 4;
        const int q4 = ((row & 1) << 1) | (row >> 1);
#pragma unroll
        for (int m = 0; m < M; ++m) {
            float su = 0.f, sw = 0.f, saa = 0.f, sab = 0.f;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const float u = dx[m][r] * sA[m][r];
                su = r == 0 ? u : su + u;
                sw = r == 0 ? sB[m][r] : sw + sB[m][r];
                saa = r == 0 ? u * dx[m][r] : __builtin_fmaf(u, dx[m][r], saa);
                sab = r == 0 ? dx[m][r] * sB[m][r] : __builtin_fmaf(dx[m][r], sB[m][r], sab);
            }
            const float k1 = -g2[m].y * g2[m].z, k2 = 2.f * k1, bb = 0.5f * g1[m].w;
            const float a0 = swap16_sum(swap32_sum(__builtin_fmaf(g1[m].z, su, bb * sw) * k2,
                                                   __builtin_fmaf(bb, su, g2[m].x * sw) * k2),
                                        swap32_sum(saa * k1, sab * k2));
            const float a1 = swap16_sum(swap32_sum(sum[m][0] * k1, sum[m][1]),
                                        swap32_sum(sum[m][2] * (g2[m].y * 0.69314718055994531f), 0.f));
            // transposed through LDS so that 16 consecutive lanes add one
            // primitive's record: the memory side takes one 64-byte line per
            // request however many of its floats it adds to (20 G lines/s)
            wave_lds_fence();
            float *out = &s_tr[li * kTrStride + q4];
            out[0] = a0;
            out[4] = q4 == 3 ? g2[m].w : a1;  // (value 7: the id)
            if constexpr (!kMfma) {
                float c4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int k = 0; k < CDIM; ++k) c4[k] = scol[m][k];
                out[8] = swap16_sum(swap32_sum(c4[0], c4[1]), swap32_sum(c4[2], c4[3]));
            }
            wave_lds_fence();
            const float *in = &s_tr[row * kTrStride];
            float val[4];
            int id[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {  // primitive 4 k + row of the group
                val[k] = in[4 * k * kTrStride + li];
                id[k] = __float_as_int(in[4 * k * kTrStride + 7]);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (grad_lane && M * (4 * k + row) + m < left && val[k] != 0.f)
                    atomic_add_f32(grad_base + (int64_t)id[k] * grad_stride, val[k]);
        }
        if constexpr (kMfma) {
            // lane -> channel li of primitives 4 row + r
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (4 * row + r >= left) continue;
                int e = q_head + 4 * row + r;
                e = e >= QN ? e - QN : e;
                const int64_t g = __float_as_int(q_geo2[e].w);
#pragma unroll
                for (int s = 0; s < NFD; ++s)
                    if (16 * s + li < CDIM && dcol[s][r] != 0.f)
                        atomic_add_f32(v_colors + g * channels + coff + 16 * s + li, dcol[s][r]);
            }
        }
        const int taken = min(left, 16 * M);
        q_count -= taken;
        q_head += taken;
        q_head = q_head >= QN ? q_head - QN : q_head;
        wave_lds_fence();
    };

    // Spans of the list, last first: all of it, or with checkpoints the
    // forward's batches [range_start + k BS, ...), each restarted from the
    // forward's T after it (for the pixels that the forward ran it for).
    const int32_t last = min(range_end - 1, wave_bin_max);
    const int32_t nspan = last < range_start ? 0 : T_ckpt ? (last - range_start) / BS + 1 : 1;
    for (int32_t sp = nspan - 1; sp >= 0; --sp) {
        const int32_t lo = range_start + (T_ckpt ? sp * BS : 0);
        const int32_t hi = T_ckpt ? list_batch_last(lo, last, BS) : last;
        if (T_ckpt) {
            if (inside && bin_final >= lo)
                px.T[lane] = (TT)T_ckpt[ckpt_slot(range_start, logical, sp, BS) * BS +
                                        sub * 64 + lane];
            wave_lds_fence();
        }
        // 64 entries at a time, back to front (lane l: entry at - l); the next
        // chunk's ids and masks are read while this one is queued and blended
        typedef typename EntryMask<SB>::type EM;
        const EM *em = static_cast<const EM *>(entry_masks);
        auto id_of = [&](const int32_t e) { return e >= lo ? flatten_ids[e] : -1; };
        auto mask_of = [&](const int32_t e) -> uint32_t { return em && e >= lo ? em[e] : ~0u; };
        int32_t g_next = id_of(hi - lane);
        uint32_t m_next = mask_of(hi - lane);
        for (int32_t at = hi; at >= lo; at -= 64) {
            const int32_t g_raw = g_next;
            const uint32_t sub_mask = m_next;
            g_next = id_of(at - 64 - lane);
            m_next = mask_of(at - 64 - lane);
            // an id outside [0, C N) (past the span's start, or from a sort that
            // gave up) is never blended
            bool hit = (uint64_t)(uint32_t)g_raw < (uint64_t)C * N && ((sub_mask >> sub) & 1u);
            if constexpr (STATS) st_staged += (uint32_t)(at - lane >= lo);
            const int64_t g = g_raw;
            float2 xy = make_float2(0.f, 0.f);
            float ca = 0.f, cb = 0.f, cc = 0.f, op = 0.f, be = 0.f;
            float4 cw = make_float4(0.f, 0.f, 0.f, 0.f);
            if (hit) {
                if (rec && wide_rec) {  // one 64-byte record per (camera, primitive), colours included
                    const float4 r0 = rec[4 * g], r1 = rec[4 * g + 1];
                    cw = rec[4 * g + 2];
                    xy = make_float2(r0.x, r0.y);
                    ca = r0.z; cb = r0.w; cc = r1.x; op = r1.y; be = r1.z;
                } else if (rec) {  // one 32-byte record per (camera, primitive)
                    const float4 r0 = rec[2 * g], r1 = rec[2 * g + 1];
                    xy = make_float2(r0.x, r0.y);
                    ca = r0.z; cb = r0.w; cc = r1.x; op = r1.y; be = r1.z;
                } else {
                    xy = reinterpret_cast<const float2 *>(means2d)[g];
                    ca = conics[g * 3]; cb = conics[g * 3 + 1]; cc = conics[g * 3 + 2];
                    op = opacities[g]; be = betas[g];
                }
                if (!em) {  // no masks from the forward: the sub-block's own test
                    float hx, hy;
                    support_box(ca, cb, cc, hx, hy);
                    // (opaque copies: the sub-block's bounds are formed here, not held in
                    // registers through the group loop)
                    uint32_t sx_o = sx0, sy_o = sy0;
                    asm volatile("" : "+s"(sx_o), "+s"(sy_o));
                    hit = subblock_mask_exact<1>(xy.x, xy.y, ca, cb, cc, hx, hy, (float)sx_o, (float)sy_o) & 1u;
                }
            }
            const uint64_t bal = __ballot(hit);
            if (hit) {
                int e = q_head + q_count + __popcll(bal & ((1ull << lane) - 1ull));
                e = e >= QN ? e - QN : e;
                // plain: no alpha near the clamp, no sigma of -0, a finite non-negative
                // beta, finite colours
                bool plain = op >= 0.f && op <= kNoClampOpacity && be >= 0.f && be < 1e30f && (ca > 0.f || cc > 0.f);
                q_geo[e] = make_float4(xy.x, xy.y, ca, 2.f * cb);  // 2b, as the forward
                q_geo2[e] = make_float4(cc, op, be, __int_as_float((int32_t)g));
                const float *cp = colors + g * channels + coff;
                if constexpr (!kMfma) {
                    if (!(rec && wide_rec))
                        cw = make_float4(cp[0], CDIM > 1 ? cp[1] : 0.f, CDIM > 2 ? cp[2] : 0.f, CDIM > 3 ? cp[3] : 0.f);
                    plain = plain && fabsf(cw.x) < 1e30f && fabsf(cw.y) < 1e30f && fabsf(cw.z) < 1e30f &&
                            (CDIM < 4 || fabsf(cw.w) < 1e30f);
                } else {
#pragma unroll
                    for (int k = 0; k < CDIM; ++k) {
                        const float c = cp[k];
                        q_col[kMfma ? k : 0][kMfma ? e : 0] = c;
                        plain = plain && fabsf(c) < 1e30f;
                    }
                }
                const uint32_t tagged = (uint32_t)(at - lane) | (plain ? kPlainBit : 0u);
                if constexpr (!kIdxInCol)
                    q_idx[e] = tagged;
                else
                    cw.w = __uint_as_float(tagged);
                if constexpr (!kMfma) q_colv[e] = cw;
            }
            q_count += __popcll(bal);
            wave_lds_fence();
            // full groups; at the span's start also the rest
            const bool flush = at - 64 < lo;
            while (q_count >= 16 * MMAX || (flush && q_count > 0)) {
                if (MMAX == 1 || q_count <= 16)
                    group(std::integral_constant<int, 1>{});
                else
                    group(std::integral_constant<int, MMAX>{});
            }
        }
    }
    if constexpr (STATS) {
        const uint32_t v[7] = {st_steps, st_live, st_valid, st_groups, st_staged, st_fast, st_empty};
#pragma unroll
        for (int q = 0; q < 7; ++q) {
            // steps, groups and their classes are wave-uniform
            const unsigned long long tot =
                (q == 0 || q == 3 || q >= 5) ? (unsigned long long)v[q] : wave_sum_u64(v[q]);
            if (stats && lane == 0 && tot) atomicAdd(stats + q, tot);
        }
        if (wg_times) {  // start, end, tile and the hardware id of the workgroup
            if (lane == 0) {
                unsigned long long *o = wg_times + 4ull * blockIdx.x;
                o[0] = t_start;
                o[1] = __builtin_amdgcn_s_memrealtime();
                o[2] = logical;
                o[3] = (unsigned long long)__builtin_amdgcn_s_getreg((31 << 11) | 4);  // HW_ID
            }
        }
    }
}

template <int TS, int CDIM>
static int launch_bwd(bool f64t, uint32_t C, uint32_t N, int64_t n_isects, uint32_t channels, uint32_t coff,
                      const float *means2d, const float *conics, const float *colors, const float *opac,
                      const float *betas, const float *bg, const uint8_t *masks, uint32_t W, uint32_t H,
                      uint32_t tw, uint32_t th, const int32_t *offs, const int32_t *flat, const float *ra,
                      const int32_t *last, const float *Tf, const float *vrc, const float *vra, float *vm2,
                      float *vcon, float *vcol, float *vop, float *vbe, const float4 *rec, float *vrec,
                      const float *ck, const uint32_t *order, const void *em, hipStream_t st) {
    const int wide = rec && raster_wide_records(channels, TS) ? 1 : 0;
    if (f64t)
        raster_bwd_kernel<TS, CDIM, true><<<xcd_grid(C, tw, th) * (TS / 8) * (TS / 8), 64, 0, st>>>(
            C, N, n_isects, channels, coff, means2d, conics, colors, opac, betas, bg, masks, W, H, tw, th, offs, flat,
            ra, last, Tf, vrc, vra, vm2, vcon, vcol, vop, vbe, rec, wide, vrec, ck, nullptr, order,
            nullptr, em);
    else
        raster_bwd_kernel<TS, CDIM, false><<<xcd_grid(C, tw, th) * (TS / 8) * (TS / 8), 64, 0, st>>>(
            C, N, n_isects, channels, coff, means2d, conics, colors, opac, betas, bg, masks, W, H, tw, th, offs, flat,
            ra, last, Tf, vrc, vra, vm2, vcon, vcol, vop, vbe, rec, wide, vrec, ck, nullptr, order,
            nullptr, em);
    UBS_LAUNCH_CHECK("raster_bwd_kernel");
    return UBS_OK;
}

template <int TS>
static int launch_bwd_chunk(int cd, bool f64t, uint32_t C, uint32_t N, int64_t n_isects, uint32_t channels,
                            uint32_t coff, const float *means2d, const float *conics, const float *colors,
                            const float *opac, const float *betas, const float *bg, const uint8_t *masks, uint32_t W,
                            uint32_t H, uint32_t tw, uint32_t th, const int32_t *offs, const int32_t *flat,
                            const float *ra, const int32_t *last, const float *Tf, const float *vrc,
                            const float *vra, float *vm2, float *vcon, float *vcol, float *vop, float *vbe,
                            const float4 *rec, float *vrec, const float *ck, const uint32_t *order, const void *em, hipStream_t st) {
#define UBS_BWD_ARGS                                                                                            \
    f64t, C, N, n_isects, channels, coff, means2d, conics, colors, opac, betas, bg, masks, W, H, tw, th, offs,  \
        flat, ra, last, Tf, vrc, vra, vm2, vcon, vcol, vop, vbe, rec, vrec, ck, order, em, st
    switch (cd) {
    case 1: return launch_bwd<TS, 1>(UBS_BWD_ARGS);
    case 2: return launch_bwd<TS, 2>(UBS_BWD_ARGS);
    case 3: return launch_bwd<TS, 3>(UBS_BWD_ARGS);
    case 4: return launch_bwd<TS, 4>(UBS_BWD_ARGS);
    case 8:
        if constexpr (TS <= 16) return launch_bwd<TS, 8>(UBS_BWD_ARGS);
        break;
    case 16:
        if constexpr (TS <= 16) return launch_bwd<TS, 16>(UBS_BWD_ARGS);
        break;
    case 32:
        if constexpr (TS <= 16) return launch_bwd<TS, 32>(UBS_BWD_ARGS);
        break;
    default:
        break;
    }
#undef UBS_BWD_ARGS
    set_error("internal: bad channel chunk %d", cd);
    return UBS_ERR_INVALID;
}

// fp64 transmittance recovery switch (process-wide, read at each call).
static int g_f64_transmittance = 0;

}  // namespace ubs

using namespace ubs;

extern "C" {

// Selects fp32 (0, default) or fp64 (1) arithmetic for the backward's
// transmittance recovery.  Not part of the reference interface.
int ubs_set_backward_fp64_transmittance(int enable) {
    g_f64_transmittance = enable ? 1 : 0;
    return UBS_OK;
}

static int raster_bwd_impl(uint32_t C, uint32_t N, int64_t n_isects, uint32_t channels, const float *means2d,
                           const float *conics, const float *colors, const float *opacities, const float *betas,
                           const float *backgrounds, const uint8_t *masks, uint32_t W, uint32_t H,
                           uint32_t tile_size, uint32_t tw, uint32_t th, const int32_t *tile_offsets,
                           const int32_t *flatten_ids, const float *render_alphas, const int32_t *last_ids,
                           const float *T_final, const float *v_render_colors, const float *v_render_alphas,
                           float *v_means2d, float *v_conics, float *v_colors, float *v_opacities, float *v_betas,
                           const float *T_ckpt, size_t ckpt_n, void *workspace, size_t workspace_bytes,
                           void *stream, const void *fwd_ws = nullptr, size_t fwd_ws_bytes = 0,
                           const void *entry_masks = nullptr) {
    hipStream_t st = as_stream(stream);
    UBS_REQUIRE(tile_size == 8 || tile_size == 16 || tile_size == 32, "tile_size must be 8, 16 or 32 (got %u)",
                tile_size);
    UBS_REQUIRE(channels >= 1, "channels must be >= 1");
    UBS_REQUIRE((uint64_t)tw * tile_size >= W && (uint64_t)th * tile_size >= H, "tile grid does not cover the image");
    UBS_REQUIRE(n_isects >= 0 && n_isects < (1ll << 31), "n_isects out of range");
    const uint64_t CN = (uint64_t)C * N;
    UBS_REQUIRE(CN == 0 || (v_means2d && v_conics && v_colors && v_opacities && v_betas), "null gradient output");
    const bool packed = workspace != nullptr && n_isects != 0 && (uint64_t)C * W * H != 0 && CN != 0;
    if (fwd_ws) {  // the forward's records and order; this workspace holds the packed gradients only
        UBS_REQUIRE(workspace, "a forward workspace needs a gradient workspace beside it");
        const size_t need = raster_workspace_bytes(C, N, 0), need_fwd = need + raster_order_bytes(C, tw, th);
        if (workspace_bytes < need || fwd_ws_bytes < need_fwd) {
            set_error("blend workspaces of %zu (gradients) and %zu (forward) bytes, %zu and %zu needed",
                      workspace_bytes, fwd_ws_bytes, need, need_fwd);
            return UBS_ERR_WORKSPACE;
        }
    } else if (workspace) {
        const size_t need = raster_workspace_bytes(C, N, 1);
        if (workspace_bytes < need) {
            set_error("blend workspace of %zu bytes, %zu needed", workspace_bytes, need);
            return UBS_ERR_WORKSPACE;
        }
    }
    const float4 *rec = nullptr;
    float *vrec = nullptr;
    const uint32_t *order = nullptr;
    const bool wide = packed && raster_wide_records(channels, tile_size);
    int e = wide ? UBS_OK : zero_async(v_colors, CN * channels * sizeof(float), st);
    if (packed && fwd_ws) {
        // the forward packed these records and wrote the tile order from the
        // same inputs: only the gradient records are cleared here
        vrec = static_cast<float *>(workspace);
        if (!e) e = zero_async(vrec, CN * (wide ? kWideRecordFloats : kRecordFloats) * sizeof(float), st);
        if (e) return e;
        rec = static_cast<const float4 *>(fwd_ws);
        order = reinterpret_cast<const uint32_t *>(static_cast<const char *>(fwd_ws) + raster_workspace_bytes(C, N, 0));
    } else if (packed) {
        // records in the first half of the workspace, packed gradients in the
        // second; the scalar gradient tensors are written by the unpack below
        float4 *r = static_cast<float4 *>(workspace);
        vrec = reinterpret_cast<float *>(static_cast<char *>(workspace) + raster_workspace_bytes(C, N, 0));
        if (!e) e = zero_async(vrec, CN * (wide ? kWideRecordFloats : kRecordFloats) * sizeof(float), st);
        if (e) return e;
        UBS_REQUIRE(means2d && conics && opacities && betas, "null pointer");
        raster_pack_kernel<<<grid_for((int64_t)CN), kThreads, 0, st>>>(CN, means2d, conics, opacities, betas, r,
                                                                       wide ? colors : nullptr, channels);
        UBS_LAUNCH_CHECK("raster_pack_kernel");
        rec = r;
        const size_t base = raster_workspace_bytes(C, N, 1);
        if (tile_offsets && workspace_bytes >= base + raster_order_bytes(C, tw, th)) {  // room for the block order
            uint32_t *o = reinterpret_cast<uint32_t *>(static_cast<char *>(workspace) + base);
            raster_block_order_kernel<<<1, kOrderThreads, 0, st>>>(C, tw, th, tile_offsets, n_isects, nullptr, o);
            UBS_LAUNCH_CHECK("raster_block_order_kernel");
            order = o;
        }
    } else {
        if (!e) e = zero_async(v_means2d, CN * 2 * sizeof(float), st);
        if (!e) e = zero_async(v_conics, CN * 3 * sizeof(float), st);
        if (!e) e = zero_async(v_opacities, CN * sizeof(float), st);
        if (!e) e = zero_async(v_betas, CN * sizeof(float), st);
        if (e) return e;
    }
    if (n_isects == 0 || (uint64_t)C * W * H == 0) return UBS_OK;
    UBS_REQUIRE((uint64_t)C * th * tw < (1ull << 31), "too many tiles");
    UBS_REQUIRE(means2d && conics && colors && opacities && betas && tile_offsets && flatten_ids && last_ids &&
                    (render_alphas || T_final) && v_render_colors,
                "null pointer");
    if (T_ckpt) {
        const size_t need = ckpt_floats(C, n_isects, tw, th, tile_size);
        if (ckpt_n < need) {
            set_error("transmittance checkpoint buffer of %zu floats, %zu needed", ckpt_n, need);
            return UBS_ERR_WORKSPACE;
        }
    }
    const bool f64t = g_f64_transmittance != 0;
    uint32_t coff = 0;
    while (coff < channels) {
        const int cd = pick_chunk(channels - coff, tile_size);
        if (tile_size == 16)
            e = launch_bwd_chunk<16>(cd, f64t, C, N, n_isects, channels, coff, means2d, conics, colors, opacities,
                                     betas, backgrounds, masks, W, H, tw, th, tile_offsets, flatten_ids,
                                     render_alphas, last_ids, T_final, v_render_colors, v_render_alphas, v_means2d,
                                     v_conics, v_colors, v_opacities, v_betas, rec, vrec, T_ckpt, order,
                                     entry_masks, st);
        else if (tile_size == 8)
            e = launch_bwd_chunk<8>(cd, f64t, C, N, n_isects, channels, coff, means2d, conics, colors, opacities,
                                    betas, backgrounds, masks, W, H, tw, th, tile_offsets, flatten_ids,
                                    render_alphas, last_ids, T_final, v_render_colors, v_render_alphas, v_means2d,
                                    v_conics, v_colors, v_opacities, v_betas, rec, vrec, T_ckpt, order,
                                     entry_masks, st);
        else
            e = launch_bwd_chunk<32>(cd, f64t, C, N, n_isects, channels, coff, means2d, conics, colors, opacities,
                                     betas, backgrounds, masks, W, H, tw, th, tile_offsets, flatten_ids,
                                     render_alphas, last_ids, T_final, v_render_colors, v_render_alphas, v_means2d,
                                     v_conics, v_colors, v_opacities, v_betas, rec, vrec, T_ckpt, order,
                                     entry_masks, st);
        if (e) return e;
        coff += (uint32_t)cd;
    }
    if (packed) {
        raster_unpack_grads_kernel<<<grid_for((int64_t)CN), kThreads, 0, st>>>(
            CN, reinterpret_cast<const float4 *>(vrec), v_means2d, v_conics, v_opacities, v_betas,
            wide ? v_colors : nullptr, channels);
        UBS_LAUNCH_CHECK("raster_unpack_grads_kernel");
    }
    return UBS_OK;
}

int ubs_rasterize_to_pixels_bwd(uint32_t C, uint32_t N, int64_t n_isects, uint32_t channels, const float *means2d,
                                const float *conics, const float *colors, const float *opacities,
                                const float *betas, const float *backgrounds, const uint8_t *masks, uint32_t W,
                                uint32_t H, uint32_t tile_size, uint32_t tw, uint32_t th,
                                const int32_t *tile_offsets, const int32_t *flatten_ids, const float *render_alphas,
                                const int32_t *last_ids, const float *T_final, const float *v_render_colors,
                                const float *v_render_alphas, float *v_means2d, float *v_conics, float *v_colors,
                                float *v_opacities, float *v_betas, void *workspace, size_t workspace_bytes,
                                void *stream) {
    return raster_bwd_impl(C, N, n_isects, channels, means2d, conics, colors, opacities, betas, backgrounds, masks, W,
                           H, tile_size, tw, th, tile_offsets, flatten_ids, render_alphas, last_ids, T_final,
                           v_render_colors, v_render_alphas, v_means2d, v_conics, v_colors, v_opacities, v_betas,
                           nullptr, 0, workspace, workspace_bytes, stream);
}

int ubs_rasterize_to_pixels_bwd_reuse(uint32_t C, uint32_t N, int64_t n_isects, uint32_t channels,
                                      const float *means2d, const float *conics, const float *colors,
                                      const float *opacities, const float *betas, const float *backgrounds,
                                      const uint8_t *masks, uint32_t W, uint32_t H, uint32_t tile_size, uint32_t tw,
                                      uint32_t th, const int32_t *tile_offsets, const int32_t *flatten_ids,
                                      const float *render_alphas, const int32_t *last_ids, const float *T_final,
                                      const float *T_ckpt, size_t ckpt_n, const float *v_render_colors,
                                      const float *v_render_alphas, float *v_means2d, float *v_conics,
                                      float *v_colors, float *v_opacities, float *v_betas, const void *fwd_workspace,
                                      size_t fwd_workspace_bytes, void *workspace, size_t workspace_bytes,
                                      void *stream) {
    UBS_REQUIRE(fwd_workspace, "null forward workspace");
    return raster_bwd_impl(C, N, n_isects, channels, means2d, conics, colors, opacities, betas, backgrounds, masks, W,
                           H, tile_size, tw, th, tile_offsets, flatten_ids, render_alphas, last_ids, T_final,
                           v_render_colors, v_render_alphas, v_means2d, v_conics, v_colors, v_opacities, v_betas,
                           T_ckpt, ckpt_n, workspace, workspace_bytes, stream, fwd_workspace, fwd_workspace_bytes);
}

int ubs_rasterize_to_pixels_bwd_keep(uint32_t C, uint32_t N, int64_t n_isects, uint32_t channels,
                                     const float *means2d, const float *conics, const float *colors,
                                     const float *opacities, const float *betas, const float *backgrounds,
                                     const uint8_t *masks, uint32_t W, uint32_t H, uint32_t tile_size, uint32_t tw,
                                     uint32_t th, const int32_t *tile_offsets, const int32_t *flatten_ids,
                                     const float *render_alphas, const int32_t *last_ids, const float *T_final,
                                     const float *T_ckpt, size_t ckpt_n, const float *v_render_colors,
                                     const float *v_render_alphas, float *v_means2d, float *v_conics,
                                     float *v_colors, float *v_opacities, float *v_betas, const void *entry_masks,
                                     size_t entry_mask_n, const void *fwd_workspace, size_t fwd_workspace_bytes,
                                     void *workspace, size_t workspace_bytes, void *stream) {
    UBS_REQUIRE(fwd_workspace, "null forward workspace");
    UBS_REQUIRE(n_isects >= 0, "n_isects out of range");
    if (entry_masks && entry_mask_n < entry_mask_bytes(n_isects, tile_size)) {
        set_error("entry masks of %zu bytes, %zu needed", entry_mask_n, entry_mask_bytes(n_isects, tile_size));
        return UBS_ERR_WORKSPACE;
    }
    return raster_bwd_impl(C, N, n_isects, channels, means2d, conics, colors, opacities, betas, backgrounds, masks, W,
                           H, tile_size, tw, th, tile_offsets, flatten_ids, render_alphas, last_ids, T_final,
                           v_render_colors, v_render_alphas, v_means2d, v_conics, v_colors, v_opacities, v_betas,
                           T_ckpt, ckpt_n, workspace, workspace_bytes, stream, fwd_workspace, fwd_workspace_bytes,
                           entry_masks);
}

int ubs_rasterize_to_pixels_bwd_ckpt(uint32_t C, uint32_t N, int64_t n_isects, uint32_t channels,
                                     const float *means2d, const float *conics, const float *colors,
                                     const float *opacities, const float *betas, const float *backgrounds,
                                     const uint8_t *masks, uint32_t W, uint32_t H, uint32_t tile_size, uint32_t tw,
                                     uint32_t th, const int32_t *tile_offsets, const int32_t *flatten_ids,
                                     const float *render_alphas, const int32_t *last_ids, const float *T_final,
                                     const float *T_ckpt, size_t ckpt_n, const float *v_render_colors,
                                     const float *v_render_alphas, float *v_means2d, float *v_conics,
                                     float *v_colors, float *v_opacities, float *v_betas, void *workspace,
                                     size_t workspace_bytes, void *stream) {
    UBS_REQUIRE(T_ckpt || n_isects == 0, "null checkpoint buffer");
    return raster_bwd_impl(C, N, n_isects, channels, means2d, conics, colors, opacities, betas, backgrounds, masks, W,
                           H, tile_size, tw, th, tile_offsets, flatten_ids, render_alphas, last_ids, T_final,
                           v_render_colors, v_render_alphas, v_means2d, v_conics, v_colors, v_opacities, v_betas,
                           T_ckpt, ckpt_n, workspace, workspace_bytes, stream);
}

#ifdef UBS_PROBE_BUILD
// Measurement build only (libubs_probe.so): the 16x16-tile, 3-channel blend
// backward with the STATS counters on the library's packed path (its
// gradients stay packed in the workspace); stats: 7 zeroed uint64.
__attribute__((visibility("default"))) int ubs_probe_raster_bwd_stats(
    uint32_t C, uint32_t N, int64_t n_isects, const float *means2d, const float *conics, const float *colors,
    const float *opacities, const float *betas, uint32_t W, uint32_t H, uint32_t tw, uint32_t th,
    const int32_t *tile_offsets, const int32_t *flatten_ids, const int32_t *last_ids, const float *T_final,
    const float *v_render_colors, const float *v_render_alphas, float *v_colors, void *workspace,
    unsigned long long *stats, void *stream) {
    hipStream_t st = as_stream(stream);
    const uint64_t CN = (uint64_t)C * N;
    float4 *r = static_cast<float4 *>(workspace);
    float *vrec = reinterpret_cast<float *>(static_cast<char *>(workspace) + raster_workspace_bytes(C, N, 0));
    int e = zero_async(v_colors, CN * 3 * sizeof(float), st);
    if (!e) e = zero_async(vrec, CN * kWideRecordFloats * sizeof(float), st);
    if (e) return e;
    raster_pack_kernel<<<grid_for((int64_t)CN), kThreads, 0, st>>>(CN, means2d, conics, opacities, betas, r,
                                                                   colors, 3);
    raster_bwd_kernel<16, 3, false, true><<<xcd_grid(C, tw, th) * 4, 64, 0, st>>>(
        C, N, n_isects, 3, 0, means2d, conics, colors, opacities, betas, nullptr, nullptr, W, H, tw, th,
        tile_offsets, flatten_ids, nullptr, last_ids, T_final, v_render_colors, v_render_alphas, nullptr, nullptr,
        v_colors, nullptr, nullptr, r, 1, vrec, nullptr, stats);
    return (int)hipGetLastError();
}

// The same backward through `order` (null: raster order) writing per
// workgroup its start, end, tile and hardware id into wg_times
// [xcd_grid * 4] (zeroed); stats may be null (timing only).
__attribute__((visibility("default"))) int ubs_probe_raster_bwd_times(
    uint32_t C, uint32_t N, int64_t n_isects, const float *means2d, const float *conics, const float *colors,
    const float *opacities, const float *betas, uint32_t W, uint32_t H, uint32_t tw, uint32_t th,
    const int32_t *tile_offsets, const int32_t *flatten_ids, const int32_t *last_ids, const float *T_final,
    const float *v_render_colors, const float *v_render_alphas, float *v_colors, void *workspace,
    const uint32_t *order, unsigned long long *stats, unsigned long long *wg_times, void *stream) {
    hipStream_t st = as_stream(stream);
    const uint64_t CN = (uint64_t)C * N;
    float4 *r = static_cast<float4 *>(workspace);
    float *vrec = reinterpret_cast<float *>(static_cast<char *>(workspace) + raster_workspace_bytes(C, N, 0));
    int e = zero_async(v_colors, CN * 3 * sizeof(float), st);
    if (!e) e = zero_async(vrec, CN * kWideRecordFloats * sizeof(float), st);
    if (e) return e;
    raster_pack_kernel<<<grid_for((int64_t)CN), kThreads, 0, st>>>(CN, means2d, conics, opacities, betas, r,
                                                                   colors, 3);
    raster_bwd_kernel<16, 3, false, true><<<xcd_grid(C, tw, th) * 4, 64, 0, st>>>(
        C, N, n_isects, 3, 0, means2d, conics, colors, opacities, betas, nullptr, nullptr, W, H, tw, th,
        tile_offsets, flatten_ids, nullptr, last_ids, T_final, v_render_colors, v_render_alphas, nullptr, nullptr,
        v_colors, nullptr, nullptr, r, 1, vrec, nullptr, stats, order, wg_times);
    return (int)hipGetLastError();
}
#endif

}  // extern "C"
