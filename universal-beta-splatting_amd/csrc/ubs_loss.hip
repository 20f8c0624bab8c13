// Image loss of the training step on gfx950: (1 - lambda) L1 + lambda (1 - SSIM)
// between rendered images and targets, forward and backward.
//
// What train.py:117-121 evaluates per view with torch's l1_loss and the
// external fused_ssim, whose arithmetic is the SSIM of utils/loss_utils.py:
// 45-80: per channel, an 11x11 Gaussian window (sigma 1.5) correlated with
// zero padding, mu1 = G*x, mu2 = G*y, s11 = G*x^2 - mu1^2, s22 = G*y^2 - mu2^2,
// s12 = G*xy - mu1 mu2, S = (2 mu1 mu2 + C1)(2 s12 + C2) /
// ((mu1^2 + mu2^2 + C1)(s11 + s22 + C2)), C1 = 0.01^2, C2 = 0.03^2, and the
// loss averages S over every pixel and channel.
//
// Images are [B, H, W, C] float32 (the rasteriser's layout; no permute).
// Pixels of up to four channels take the streaming kernels below; wider ones one
// workgroup per 16x16 pixel tile and (image, channel): the 26x26 input
// halo is staged in LDS and the window is applied separably (rows, then
// columns).  The forward writes, per element, dL/dmu1, dL/ds11 and dL/ds12
// (the derivatives of the averaged SSIM term w.r.t. the three filtered maps
// the pixel's S depends on) into the workspace, and one partial sum of S and
// of |x - y| per workgroup; a one-block kernel adds those up in a fixed
// order.  The backward correlates the three derivative maps with the same
// window (the adjoint of a symmetric correlation) and adds the L1 term:
//   dL/dx = G*dmu1 + 2 x G*ds11 + y G*ds12 + (1 - lambda) sign(x - y) / n.
// With lambda = 0 both directions are one grid-stride float4 pass.
#pragma clang fp contract(off)

#include <algorithm>
#include <cmath>

#include "ubs_common.h"

namespace ubs {

constexpr int kLossTile = 16;
constexpr int kWin = 11;
constexpr int kHalo = kWin / 2;                 // 5
constexpr int kSpan = kLossTile + 2 * kHalo;    // 26
constexpr float kC1 = 0.01f * 0.01f;
constexpr float kC2 = 0.03f * 0.03f;

// Tiles of a launch (256 threads each, fewer than 2^32 in all).
constexpr int64_t kMaxTiles = 1ll << 24;

struct LossLayout {
    size_t partial_off, dmaps_off, total;
    int64_t blocks;
};

// The strips of the streaming kernels: 256 of a row's W C values wide, and
// chunks x 11 input rows (10 fewer output rows) high.
constexpr int kStripCols = 256;
constexpr int kStripBlocks = 700;

struct StripShape {
    int64_t cols, strips;  // column blocks, strips of an image
    int chunks;
    int64_t rows() const { return (int64_t)chunks * kWin - 2 * kHalo; }
    int64_t blocks() const { return cols * strips; }
};

// Longer strips repeat less of their halo (4 chunks: 44 input rows for 34 output
// rows, 2: 22 for 12), shorter ones fill the chip.  512 workgroups of the forward
// and 768 of the backward are resident, and a few past a multiple of either take
// another round, so the time is not monotone in the length (1080p, three
// channels, forward and backward with the host's calls, by chunks: 2, 2070
// workgroups: 162 us; 3, 1081: 149; 4, 736: 127; 5, 552: 147; 6, 460: 134; 8,
// 322: 165).  The longest with 700 workgroups or more is the best of them there and
// within 20% of the best at every size measured from 256x256 to 3840x2160 (720p: 91
// us with 2 chunks, 76 with 3; 2560x1440: 238 with 8, 208 with 7).
static StripShape strip_shape(int64_t B, int64_t H, int64_t W, int64_t C) {
    StripShape s{};
    s.cols = (W * C + kStripCols - 1) / kStripCols;
    for (s.chunks = 8;; --s.chunks) {
        s.strips = (H + s.rows() - 1) / s.rows();
        if (s.chunks == 2 || s.blocks() * B >= kStripBlocks) return s;
    }
}

// Pixels of up to four channels stream; wider ones (whose halo of 10 C values
// would not fit) take the tiles.  A column's byte offset in its row has 32 bits.
static bool streams(int64_t B, int64_t H, int64_t W, int64_t C) {
    return C <= 4 && W * C < (1ll << 30) - 4096 && strip_shape(B, H, W, C).blocks() < (1ll << 31) && B < 65536;
}

static LossLayout loss_layout(int64_t B, int64_t H, int64_t W, int64_t C) {
    LossLayout L{};
    const int64_t tx = (W + kLossTile - 1) / kLossTile, ty = (H + kLossTile - 1) / kLossTile;
    L.blocks = std::max<int64_t>(streams(B, H, W, C) ? strip_shape(B, H, W, C).blocks() * B : tx * ty * B * C, 1);
    L.partial_off = 0;
    // also the L1 pass's 1024 blocks, and the tiles of a misaligned one
    size_t off = (size_t)std::max<int64_t>(std::max<int64_t>(L.blocks, tx * ty * B * C), 1024) * 2 * sizeof(float);
    off = (off + 255) & ~(size_t)255;
    L.dmaps_off = off;
    off += (size_t)3 * B * H * W * C * sizeof(float);
    L.total = (off + 255) & ~(size_t)255;
    return L;
}

// The normalised 11-tap Gaussian of loss_utils.py:26-33 (float weights of
// exp(-(k-5)^2 / 4.5), divided by their float sum).
struct GaussWin {
    float g[kWin];
};

static GaussWin gauss_window() {
    GaussWin w;
    float s = 0.f;
    for (int k = 0; k < kWin; ++k) {
        const double d = (double)(k - kHalo);
        w.g[k] = (float)std::exp(-(d * d) / (2.0 * 1.5 * 1.5));
    }
    for (int k = 0; k < kWin; ++k) s += w.g[k];
    for (int k = 0; k < kWin; ++k) w.g[k] /= s;
    return w;
}

__device__ __forceinline__ int64_t elem(int64_t b, int64_t i, int64_t j, int64_t c, int64_t H, int64_t W,
                                        int64_t C) {
    return ((b * H + i) * W + j) * C + c;
}

// Block sums of two floats (256 threads) -> thread 0.
__device__ __forceinline__ void block_sum2(float &a, float &b, float *lds) {
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_xor(a, o, 64);
        b += __shfl_xor(b, o, 64);
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        lds[2 * w] = a;
        lds[2 * w + 1] = b;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        a = (lds[0] + lds[2]) + (lds[4] + lds[6]);
        b = (lds[1] + lds[3]) + (lds[5] + lds[7]);
    }
}

template <bool SSIM>
__global__ __launch_bounds__(256) void loss_fwd_kernel(int64_t B, int64_t H, int64_t W, int64_t C,
                                                       const float *__restrict__ x, const float *__restrict__ y,
                                                       GaussWin win, float lambda, float inv_n,
                                                       float *__restrict__ partial, float *__restrict__ dmaps) {
    __shared__ float sx[kSpan][kSpan + 1], sy[kSpan][kSpan + 1];
    __shared__ float h[5][kSpan][kLossTile + 1];
    __shared__ float red[8];
    const int64_t tiles_x = (W + kLossTile - 1) / kLossTile;
    const int64_t bc = blockIdx.y;  // image * C + channel
    const int64_t b = bc / C, c = bc % C;
    const int64_t i0 = (int64_t)(blockIdx.x / tiles_x) * kLossTile, j0 = (int64_t)(blockIdx.x % tiles_x) * kLossTile;
    const int tid = threadIdx.x;
    const int ti = tid / kLossTile, tj = tid % kLossTile;
    const int64_t i = i0 + ti, j = j0 + tj;
    const bool inside = i < H && j < W;
    float s_sum = 0.f, l1_sum = 0.f;
    if constexpr (SSIM) {
        for (int k = tid; k < kSpan * kSpan; k += 256) {
            const int r = k / kSpan, q = k % kSpan;
            const int64_t ii = i0 - kHalo + r, jj = j0 - kHalo + q;
            const bool ok = ii >= 0 && ii < H && jj >= 0 && jj < W;  // zero padding
            sx[r][q] = ok ? x[elem(b, ii, jj, c, H, W, C)] : 0.f;
            sy[r][q] = ok ? y[elem(b, ii, jj, c, H, W, C)] : 0.f;
        }
        __syncthreads();
        // rows: the five products filtered along j for all 26 halo rows
        for (int k = tid; k < kSpan * kLossTile; k += 256) {
            const int r = k / kLossTile, q = k % kLossTile;
            float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f, a4 = 0.f;
#pragma unroll
            for (int t = 0; t < kWin; ++t) {
                const float g = win.g[t], u = sx[r][q + t], v = sy[r][q + t];
                a0 += g * u;
                a1 += g * v;
                a2 += g * (u * u);
                a3 += g * (v * v);
                a4 += g * (u * v);
            }
            h[0][r][q] = a0;
            h[1][r][q] = a1;
            h[2][r][q] = a2;
            h[3][r][q] = a3;
            h[4][r][q] = a4;
        }
        __syncthreads();
        float m1 = 0.f, m2 = 0.f, e11 = 0.f, e22 = 0.f, e12 = 0.f;
#pragma unroll
        for (int t = 0; t < kWin; ++t) {
            const float g = win.g[t];
            m1 += g * h[0][ti + t][tj];
            m2 += g * h[1][ti + t][tj];
            e11 += g * h[2][ti + t][tj];
            e22 += g * h[3][ti + t][tj];
            e12 += g * h[4][ti + t][tj];
        }
        if (inside) {
            const float mu11 = m1 * m1, mu22 = m2 * m2, mu12 = m1 * m2;
            const float s11 = e11 - mu11, s22 = e22 - mu22, s12 = e12 - mu12;
            const float A1 = 2.f * mu12 + kC1, A2 = 2.f * s12 + kC2;
            const float B1 = mu11 + mu22 + kC1, B2 = s11 + s22 + kC2;
            const float D = B1 * B2;
            const float S = (A1 * A2) / D;
            s_sum = S;
            // derivatives of S w.r.t. mu1, E[x^2] and E[xy] (loss_utils.py:56-80)
            const float dmu1 = (2.f * m2 * (A2 - A1) - 2.f * m1 * S * (B2 - B1)) / D;
            const float ds11 = -S / B2;
            const float ds12 = 2.f * A1 / D;
            const float k = -lambda * inv_n;  // d loss / d S at every element
            const int64_t e = elem(b, i, j, c, H, W, C), n_el = B * H * W * C;
            dmaps[e] = k * dmu1;
            dmaps[n_el + e] = k * ds11;
            dmaps[2 * n_el + e] = k * ds12;
        }
    }
    if (inside) l1_sum = fabsf(x[elem(b, i, j, c, H, W, C)] - y[elem(b, i, j, c, H, W, C)]);
    block_sum2(s_sum, l1_sum, red);
    if (tid == 0) {
        const int64_t blk = bc * gridDim.x + blockIdx.x;
        partial[2 * blk] = s_sum;
        partial[2 * blk + 1] = l1_sum;
    }
}

// The streaming kernels (pixels of up to four channels).  A row of the image is
// W C consecutive values and the window's taps along it are C values apart, so a
// thread takes one of 256 consecutive values (coalesced, whatever the channel)
// and walks down the rows: 11 input rows at a time are staged in LDS with a halo
// of 5 C values on either side, a row is filtered along itself from there, and
// the last 11 filtered rows stay in registers for the filter across rows (the
// loop over 11 rows is unrolled, so a row's place in the ring is a constant).
// Bound by VALU issue and its dependent chains at 2-3 waves per SIMD (the ring and
// the chunk under way take 170-210 registers): about 160 instructions an element
// in the forward, 1.3 times for the halo rows.  Forward and backward at 1080p,
// three channels: 66 and 54 us, where tiles of 16 x 16 pixels of one channel, which
// read 2.6 times their pixels at a stride of C values and pass every filtered row
// through LDS, took 124 and 111.  (Held to 128 registers: 88 and 75.)
//
// 11 rows of M images: a thread holds its own column's values and its share of the
// two halos' (11 x 10 C values an image).  A row's address is the same for the
// whole workgroup, so that a load needs only the column's 32-bit offset.
template <int C, int M>
struct Chunk {
    static constexpr int kPad = kHalo * C, kRow = kStripCols + 2 * kPad;
    static constexpr int kHaloAll = M * kWin * 2 * kPad, kPer = (kHaloAll + kStripCols - 1) / kStripCols;
    float own[M][kWin], halo[kPer];

    __device__ __forceinline__ void load(const float *const (&img)[M], int64_t first, int64_t H, int64_t len,
                                         int64_t f0) {
        const int tid = threadIdx.x;
        const bool col = f0 + tid < len;
        const uint32_t off = (uint32_t)(col ? f0 + tid : 0) * 4u;
#pragma unroll
        for (int r = 0; r < kWin; ++r) {
            const int64_t i = first + r;
            const bool row = i >= 0 && i < H;  // zero padding
            const int64_t at = (row ? i : 0) * len;
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const float v = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(img[m] + at) + off);
                own[m][r] = row && col ? v : 0.f;
            }
        }
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const int k = tid + u * kStripCols, m = k / (kWin * 2 * kPad), q = k % (2 * kPad);
            const int64_t i = first + k / (2 * kPad) % kWin, f = q < kPad ? f0 - kPad + q : f0 + kStripCols + q - kPad;
            const bool ok = k < kHaloAll && i >= 0 && i < H && f >= 0 && f < len;
            const float *const src = m == 0 ? img[0] : m == 1 || M == 2 ? img[M > 1 ? 1 : 0] : img[M - 1];
            halo[u] = ok ? src[i * len + f] : 0.f;
        }
    }
    __device__ __forceinline__ void store(float (&s)[M][kWin][kRow]) const {
        const int tid = threadIdx.x;
#pragma unroll
        for (int r = 0; r < kWin; ++r)
#pragma unroll
            for (int m = 0; m < M; ++m) s[m][r][kPad + tid] = own[m][r];
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const int k = tid + u * kStripCols, q = k % (2 * kPad);
            if (k < kHaloAll) s[k / (kWin * 2 * kPad)][k / (2 * kPad) % kWin][q < kPad ? q : q + kStripCols] = halo[u];
        }
    }
};

template <int C>
__global__ __launch_bounds__(kStripCols, 2) void ssim_fwd_kernel(int64_t H, int64_t len, int64_t cols, int chunks,
                                                              const float *__restrict__ x,
                                                              const float *__restrict__ y, GaussWin win, float k,
                                                              int64_t n_el, float *__restrict__ partial,
                                                              float *__restrict__ dmaps) {
    __shared__ float sxy[2][kWin][Chunk<C, 2>::kRow];
    __shared__ double red[2][kStripCols / 64];
    const int tid = threadIdx.x;
    const int64_t strip = blockIdx.x / cols, f0 = (int64_t)(blockIdx.x % cols) * kStripCols, f = f0 + tid;
    const uint32_t f32 = (uint32_t)f;
    const int64_t rows = (int64_t)chunks * kWin - 2 * kHalo, i0 = strip * rows;
    const int64_t img = (int64_t)blockIdx.y * H * len;
    x += img;
    y += img;
    dmaps += img;
    float h0[kWin], h1[kWin], h2[kWin], h3[kWin], h4[kWin];  // the last 11 filtered rows
    const float *const both[2] = {x, y};
    Chunk<C, 2> next;  // (loaded while the chunk before it is filtered)
    next.load(both, i0 - kHalo, H, len, f0);
    double s_sum = 0.0, l1_sum = 0.0;
    for (int ch = 0; ch < chunks; ++ch) {
        __syncthreads();
        next.store(sxy);
        __syncthreads();
        const int64_t ir = i0 - kHalo + (int64_t)ch * kWin;  // image row of the chunk's first
        if (ch + 1 < chunks) next.load(both, ir + kWin, H, len, f0);
        float s_part = 0.f, l1_part = 0.f;
#pragma unroll
        for (int r = 0; r < kWin; ++r) {
            __builtin_amdgcn_sched_barrier(0);
            float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f, a4 = 0.f;
#pragma unroll
            for (int t = 0; t < kWin; ++t) {
                const float g = win.g[t], u = sxy[0][r][tid + t * C], v = sxy[1][r][tid + t * C];
                const float gu = g * u, gv = g * v;
                a0 += gu;
                a1 += gv;
                a2 = __builtin_fmaf(gu, u, a2);
                a3 = __builtin_fmaf(gv, v, a3);
                a4 = __builtin_fmaf(gu, v, a4);
                if (t == kHalo && ir + r >= i0 && ir + r < i0 + rows) l1_part += fabsf(u - v);  // (0 outside the image)
            }
            h0[r] = a0;
            h1[r] = a1;
            h2[r] = a2;
            h3[r] = a3;
            h4[r] = a4;
            if (ch == 0 && r < kWin - 1) continue;  // the first output row needs 11
            float m1 = 0.f, m2 = 0.f, e11 = 0.f, e22 = 0.f, e12 = 0.f;
#pragma unroll
            for (int t = 0; t < kWin; ++t) {
                constexpr int n = kWin;
                const float g = win.g[t];
                const int q = (r + 1 + t) % n;  // oldest first
                m1 = __builtin_fmaf(g, h0[q], m1);
                m2 = __builtin_fmaf(g, h1[q], m2);
                e11 = __builtin_fmaf(g, h2[q], e11);
                e22 = __builtin_fmaf(g, h3[q], e22);
                e12 = __builtin_fmaf(g, h4[q], e12);
            }
            const int64_t i = ir + r - kHalo;  // the output row
            if (i < H && f < len) {
                const float mu11 = m1 * m1, mu22 = m2 * m2, mu12 = m1 * m2;
                const float s11 = e11 - mu11, s22 = e22 - mu22, s12 = e12 - mu12;
                const float A1 = 2.f * mu12 + kC1, A2 = 2.f * s12 + kC2;
                const float B1 = mu11 + mu22 + kC1, B2 = s11 + s22 + kC2;
                const float D = B1 * B2;
                const float Sv = (A1 * A2) / D;
                s_part += Sv;
                // derivatives of S w.r.t. mu1, E[x^2] and E[xy] (loss_utils.py:56-80)
                const float dmu1 = (2.f * m2 * (A2 - A1) - 2.f * m1 * Sv * (B2 - B1)) / D;
                const float ds11 = -Sv / B2;
                const float ds12 = 2.f * A1 / D;
                float *const d = dmaps + i * len;
                d[f32] = k * dmu1;
                d[n_el + f32] = k * ds11;
                d[2 * n_el + f32] = k * ds12;
            }
        }
        s_sum += (double)s_part;
        l1_sum += (double)l1_part;
    }
    if (f >= len) l1_sum = 0.0;  // (another strip's halo)
    for (int o = 32; o > 0; o >>= 1) {
        s_sum += __shfl_xor(s_sum, o, 64);
        l1_sum += __shfl_xor(l1_sum, o, 64);
    }
    if ((tid & 63) == 0) {
        red[0][tid >> 6] = s_sum;
        red[1][tid >> 6] = l1_sum;
    }
    __syncthreads();
    if (tid == 0) {
        const int64_t blk = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
        partial[2 * blk] = (float)((red[0][0] + red[0][1]) + (red[0][2] + red[0][3]));
        partial[2 * blk + 1] = (float)((red[1][0] + red[1][1]) + (red[1][2] + red[1][3]));
    }
}

template <int C>
__global__ __launch_bounds__(kStripCols, 3) void ssim_bwd_kernel(int64_t H, int64_t len, int64_t cols, int chunks,
                                                              const float *__restrict__ x,
                                                              const float *__restrict__ y, GaussWin win, float l1,
                                                              int64_t n_el, const float *__restrict__ v_loss,
                                                              const float *__restrict__ dmaps,
                                                              float *__restrict__ v_x) {
    __shared__ float sd[3][kWin][Chunk<C, 3>::kRow];
    const int tid = threadIdx.x;
    const int64_t strip = blockIdx.x / cols, f0 = (int64_t)(blockIdx.x % cols) * kStripCols, f = f0 + tid;
    const uint32_t f32 = (uint32_t)f;
    const int64_t i0 = strip * ((int64_t)chunks * kWin - 2 * kHalo);
    const int64_t img = (int64_t)blockIdx.y * H * len;
    x += img;
    y += img;
    v_x += img;
    dmaps += img;
    const float vl = v_loss[0];
    float h[3][kWin];
    const float *const maps[3] = {dmaps, dmaps + n_el, dmaps + 2 * n_el};
    Chunk<C, 3> next;
    next.load(maps, i0 - kHalo, H, len, f0);
    for (int ch = 0; ch < chunks; ++ch) {
        __syncthreads();
        next.store(sd);
        __syncthreads();
        const int64_t ir = i0 - kHalo + (int64_t)ch * kWin;
        if (ch + 1 < chunks) next.load(maps, ir + kWin, H, len, f0);
#pragma unroll
        for (int r = 0; r < kWin; ++r) {
            __builtin_amdgcn_sched_barrier(0);
            float a[3] = {0.f, 0.f, 0.f};
#pragma unroll
            for (int t = 0; t < kWin; ++t)
#pragma unroll
                for (int m = 0; m < 3; ++m) a[m] = __builtin_fmaf(win.g[t], sd[m][r][tid + t * C], a[m]);
#pragma unroll
            for (int m = 0; m < 3; ++m) h[m][r] = a[m];
            if (ch == 0 && r < kWin - 1) continue;
            float b[3] = {0.f, 0.f, 0.f};
#pragma unroll
            for (int t = 0; t < kWin; ++t)
#pragma unroll
                for (int m = 0; m < 3; ++m) b[m] = __builtin_fmaf(win.g[t], h[m][(r + 1 + t) % kWin], b[m]);
            const int64_t i = ir + r - kHalo;
            if (i < H && f < len) {
                const int64_t at = i * len;
                const float xv = x[at + f32], yv = y[at + f32], d = xv - yv;
                const float sgn = d > 0.f ? 1.f : (d < 0.f ? -1.f : 0.f);
                v_x[at + f32] = vl * (l1 * sgn + (b[0] + 2.f * xv * b[1] + yv * b[2]));
            }
        }
    }
}

// L1 only: a grid-stride pass over float4s (plus a scalar tail), one partial
// sum of |x - y| per workgroup.
constexpr int kL1Blocks = 1024;

__global__ __launch_bounds__(256) void l1_fwd_kernel(int64_t n, const float *__restrict__ x,
                                                     const float *__restrict__ y, float *__restrict__ partial) {
    __shared__ float red[8];
    const int64_t n4 = n / 4;
    const float4 *x4 = reinterpret_cast<const float4 *>(x), *y4 = reinterpret_cast<const float4 *>(y);
    float acc = 0.f, dummy = 0.f;
    for (int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x; k < n4; k += (int64_t)gridDim.x * 256) {
        const float4 a = x4[k], b = y4[k];
        acc += (fabsf(a.x - b.x) + fabsf(a.y - b.y)) + (fabsf(a.z - b.z) + fabsf(a.w - b.w));
    }
    if (blockIdx.x == 0 && threadIdx.x < n - 4 * n4) acc += fabsf(x[4 * n4 + threadIdx.x] - y[4 * n4 + threadIdx.x]);
    block_sum2(dummy, acc, red);
    if (threadIdx.x == 0) {
        partial[2 * blockIdx.x] = 0.f;
        partial[2 * blockIdx.x + 1] = acc;
    }
}

__global__ __launch_bounds__(256) void l1_bwd_kernel(int64_t n, const float *__restrict__ x,
                                                     const float *__restrict__ y, float inv_n,
                                                     const float *__restrict__ v_loss, float *__restrict__ v_x) {
    const float s = v_loss[0] * inv_n;
    auto sg = [s](float d) { return d > 0.f ? s : (d < 0.f ? -s : 0.f); };
    const int64_t n4 = n / 4;
    const float4 *x4 = reinterpret_cast<const float4 *>(x), *y4 = reinterpret_cast<const float4 *>(y);
    float4 *v4 = reinterpret_cast<float4 *>(v_x);
    for (int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x; k < n4; k += (int64_t)gridDim.x * 256) {
        const float4 a = x4[k], b = y4[k];
        v4[k] = make_float4(sg(a.x - b.x), sg(a.y - b.y), sg(a.z - b.z), sg(a.w - b.w));
    }
    if (blockIdx.x == 0 && threadIdx.x < n - 4 * n4) {
        const int64_t e = 4 * n4 + threadIdx.x;
        v_x[e] = sg(x[e] - y[e]);
    }
}

// loss = (1 - lambda) sum|x - y| / n + lambda (1 - sum S / n), the block
// partials added in a fixed order (double accumulators).
__global__ void loss_finish_kernel(int64_t blocks, const float *__restrict__ partial, float lambda, double n,
                                   int ssim, float *__restrict__ loss) {
    __shared__ double s[2][256];
    double a = 0.0, l = 0.0;
    for (int64_t k = threadIdx.x; k < blocks; k += 256) {
        a += (double)partial[2 * k];
        l += (double)partial[2 * k + 1];
    }
    s[0][threadIdx.x] = a;
    s[1][threadIdx.x] = l;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            s[0][threadIdx.x] += s[0][threadIdx.x + o];
            s[1][threadIdx.x] += s[1][threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double l1 = s[1][0] / n;
        const double ssim_term = ssim ? (1.0 - s[0][0] / n) : 0.0;
        loss[0] = (float)((1.0 - (double)lambda) * l1 + (double)lambda * ssim_term);
    }
}

template <bool SSIM>
__global__ __launch_bounds__(256) void loss_bwd_kernel(int64_t B, int64_t H, int64_t W, int64_t C,
                                                       const float *__restrict__ x, const float *__restrict__ y,
                                                       GaussWin win, float lambda, float inv_n,
                                                       const float *__restrict__ v_loss,
                                                       const float *__restrict__ dmaps, float *__restrict__ v_x) {
    __shared__ float sd[3][kSpan][kSpan + 1];
    __shared__ float h[3][kSpan][kLossTile + 1];
    const int64_t tiles_x = (W + kLossTile - 1) / kLossTile;
    const int64_t bc = blockIdx.y;
    const int64_t b = bc / C, c = bc % C;
    const int64_t i0 = (int64_t)(blockIdx.x / tiles_x) * kLossTile, j0 = (int64_t)(blockIdx.x % tiles_x) * kLossTile;
    const int tid = threadIdx.x;
    const int ti = tid / kLossTile, tj = tid % kLossTile;
    const int64_t i = i0 + ti, j = j0 + tj;
    const bool inside = i < H && j < W;
    const int64_t n_el = B * H * W * C;
    float gm = 0.f, g11 = 0.f, g12 = 0.f;
    if constexpr (SSIM) {
        for (int k = tid; k < kSpan * kSpan; k += 256) {
            const int r = k / kSpan, q = k % kSpan;
            const int64_t ii = i0 - kHalo + r, jj = j0 - kHalo + q;
            const bool ok = ii >= 0 && ii < H && jj >= 0 && jj < W;  // no S outside the image
            const int64_t e = ok ? elem(b, ii, jj, c, H, W, C) : 0;
            sd[0][r][q] = ok ? dmaps[e] : 0.f;
            sd[1][r][q] = ok ? dmaps[n_el + e] : 0.f;
            sd[2][r][q] = ok ? dmaps[2 * n_el + e] : 0.f;
        }
        __syncthreads();
        for (int k = tid; k < kSpan * kLossTile; k += 256) {
            const int r = k / kLossTile, q = k % kLossTile;
            float a0 = 0.f, a1 = 0.f, a2 = 0.f;
#pragma unroll
            for (int t = 0; t < kWin; ++t) {
                const float g = win.g[t];
                a0 += g * sd[0][r][q + t];
                a1 += g * sd[1][r][q + t];
                a2 += g * sd[2][r][q + t];
            }
            h[0][r][q] = a0;
            h[1][r][q] = a1;
            h[2][r][q] = a2;
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < kWin; ++t) {
            const float g = win.g[t];
            gm += g * h[0][ti + t][tj];
            g11 += g * h[1][ti + t][tj];
            g12 += g * h[2][ti + t][tj];
        }
    }
    if (!inside) return;
    const int64_t e = elem(b, i, j, c, H, W, C);
    const float xv = x[e], yv = y[e], dxy = xv - yv;
    const float sgn = dxy > 0.f ? 1.f : (dxy < 0.f ? -1.f : 0.f);
    float g = (1.f - lambda) * inv_n * sgn;
    if constexpr (SSIM) g += gm + 2.f * xv * g11 + yv * g12;
    v_x[e] = v_loss[0] * g;
}

}  // namespace ubs

using namespace ubs;

extern "C" {

size_t ubs_image_loss_workspace_bytes(int64_t B, int64_t H, int64_t W, int64_t C) {
    return loss_layout(B, H, W, C).total;
}

int ubs_image_loss_fwd(int64_t B, int64_t H, int64_t W, int64_t C, const float *img, const float *gt,
                       float lambda_dssim, float *loss, void *workspace, size_t workspace_bytes, void *stream) {
    UBS_REQUIRE(B >= 0 && H >= 0 && W >= 0 && C >= 0, "negative size");
    UBS_REQUIRE(lambda_dssim >= 0.f && lambda_dssim <= 1.f, "lambda_dssim must be in [0, 1]");
    UBS_REQUIRE(loss, "null loss output");
    hipStream_t st = as_stream(stream);
    const int64_t n = B * H * W * C;
    UBS_REQUIRE(n > 0, "empty image");
    UBS_REQUIRE(img && gt, "null pointer");
    const LossLayout L = loss_layout(B, H, W, C);
    if (!workspace || workspace_bytes < L.total) {
        set_error("loss workspace too small (%zu < %zu)", workspace_bytes, L.total);
        return UBS_ERR_WORKSPACE;
    }
    const int64_t tiles = ((W + kLossTile - 1) / kLossTile) * ((H + kLossTile - 1) / kLossTile);
    UBS_REQUIRE(tiles < (1ll << 31) && B * C < 65536, "image batch too large");
    char *ws = static_cast<char *>(workspace);
    float *partial = reinterpret_cast<float *>(ws + L.partial_off);
    float *dmaps = reinterpret_cast<float *>(ws + L.dmaps_off);
    const bool ssim = lambda_dssim > 0.f;
    const bool aligned = (reinterpret_cast<uintptr_t>(img) % 16 == 0) && (reinterpret_cast<uintptr_t>(gt) % 16 == 0);
    if (!ssim && aligned) {
        const unsigned nb = (unsigned)std::min<int64_t>(kL1Blocks, std::max<int64_t>(1, (n / 4 + 255) / 256));
        l1_fwd_kernel<<<nb, 256, 0, st>>>(n, img, gt, partial);
        UBS_LAUNCH_CHECK("l1_fwd_kernel");
        loss_finish_kernel<<<1, 256, 0, st>>>(nb, partial, lambda_dssim, (double)n, 0, loss);
        UBS_LAUNCH_CHECK("loss_finish_kernel");
        return UBS_OK;
    }
    const dim3 grid((unsigned)tiles, (unsigned)(B * C));
    const GaussWin win = gauss_window();
    UBS_REQUIRE((ssim && streams(B, H, W, C)) || tiles < kMaxTiles, "image too large");
    if (ssim && streams(B, H, W, C)) {
        const StripShape s = strip_shape(B, H, W, C);
        const dim3 g((unsigned)s.blocks(), (unsigned)B);
        const float k = -lambda_dssim * (1.f / (float)n);  // d loss / d S at every element
#define UBS_SSIM_FWD(K)                                                                                              \
    case K:                                                                                                          \
        ssim_fwd_kernel<K><<<g, kStripCols, 0, st>>>(H, W * C, s.cols, s.chunks, img, gt, win, k, n, partial, dmaps); \
        break;
        switch (C) { UBS_SSIM_FWD(1) UBS_SSIM_FWD(2) UBS_SSIM_FWD(3) UBS_SSIM_FWD(4) }
#undef UBS_SSIM_FWD
        UBS_LAUNCH_CHECK("ssim_fwd_kernel");
        loss_finish_kernel<<<1, 256, 0, st>>>(L.blocks, partial, lambda_dssim, (double)n, 1, loss);
        UBS_LAUNCH_CHECK("loss_finish_kernel");
        return UBS_OK;
    }
    if (ssim)
        loss_fwd_kernel<true><<<grid, 256, 0, st>>>(B, H, W, C, img, gt, win, lambda_dssim, 1.f / (float)n, partial,
                                                    dmaps);
    else
        loss_fwd_kernel<false><<<grid, 256, 0, st>>>(B, H, W, C, img, gt, win, lambda_dssim, 1.f / (float)n,
                                                     partial, dmaps);
    UBS_LAUNCH_CHECK("loss_fwd_kernel");
    loss_finish_kernel<<<1, 256, 0, st>>>(tiles * B * C, partial, lambda_dssim, (double)n, ssim ? 1 : 0, loss);
    UBS_LAUNCH_CHECK("loss_finish_kernel");
    return UBS_OK;
}

int ubs_image_loss_bwd(int64_t B, int64_t H, int64_t W, int64_t C, const float *img, const float *gt,
                       float lambda_dssim, const float *v_loss, const void *workspace, size_t workspace_bytes,
                       float *v_img, void *stream) {
    UBS_REQUIRE(B >= 0 && H >= 0 && W >= 0 && C >= 0, "negative size");
    UBS_REQUIRE(lambda_dssim >= 0.f && lambda_dssim <= 1.f, "lambda_dssim must be in [0, 1]");
    hipStream_t st = as_stream(stream);
    const int64_t n = B * H * W * C;
    UBS_REQUIRE(n > 0, "empty image");
    UBS_REQUIRE(img && gt && v_loss && v_img, "null pointer");
    const LossLayout L = loss_layout(B, H, W, C);
    if (!workspace || workspace_bytes < L.total) {
        set_error("loss workspace too small (%zu < %zu)", workspace_bytes, L.total);
        return UBS_ERR_WORKSPACE;
    }
    const int64_t tiles = ((W + kLossTile - 1) / kLossTile) * ((H + kLossTile - 1) / kLossTile);
    UBS_REQUIRE(tiles < (1ll << 31) && B * C < 65536, "image batch too large");
    const float *dmaps = reinterpret_cast<const float *>(static_cast<const char *>(workspace) + L.dmaps_off);
    const bool aligned = (reinterpret_cast<uintptr_t>(img) % 16 == 0) && (reinterpret_cast<uintptr_t>(gt) % 16 == 0) &&
                         (reinterpret_cast<uintptr_t>(v_img) % 16 == 0);
    if (lambda_dssim == 0.f && aligned) {
        const unsigned nb = (unsigned)std::min<int64_t>(kL1Blocks, std::max<int64_t>(1, (n / 4 + 255) / 256));
        l1_bwd_kernel<<<nb, 256, 0, st>>>(n, img, gt, 1.f / (float)n, v_loss, v_img);
        UBS_LAUNCH_CHECK("l1_bwd_kernel");
        return UBS_OK;
    }
    const dim3 grid((unsigned)tiles, (unsigned)(B * C));
    const GaussWin win = gauss_window();
    UBS_REQUIRE((lambda_dssim > 0.f && streams(B, H, W, C)) || tiles < kMaxTiles, "image too large");
    if (lambda_dssim > 0.f && streams(B, H, W, C)) {
        const StripShape s = strip_shape(B, H, W, C);
        const dim3 g((unsigned)s.blocks(), (unsigned)B);
        const float l1 = (1.f - lambda_dssim) * (1.f / (float)n);
#define UBS_SSIM_BWD(K)                                                                                           \
    case K:                                                                                                       \
        ssim_bwd_kernel<K><<<g, kStripCols, 0, st>>>(H, W * C, s.cols, s.chunks, img, gt, win, l1, n, v_loss,     \
                                                     dmaps, v_img);                                               \
        break;
        switch (C) { UBS_SSIM_BWD(1) UBS_SSIM_BWD(2) UBS_SSIM_BWD(3) UBS_SSIM_BWD(4) }
#undef UBS_SSIM_BWD
        UBS_LAUNCH_CHECK("ssim_bwd_kernel");
        return UBS_OK;
    }
    if (lambda_dssim > 0.f)
        loss_bwd_kernel<true><<<grid, 256, 0, st>>>(B, H, W, C, img, gt, win, lambda_dssim, 1.f / (float)n, v_loss,
                                                    dmaps, v_img);
    else
        loss_bwd_kernel<false><<<grid, 256, 0, st>>>(B, H, W, C, img, gt, win, lambda_dssim, 1.f / (float)n, v_loss,
                                                     dmaps, v_img);
    UBS_LAUNCH_CHECK("loss_bwd_kernel");
    return UBS_OK;
}

}  // extern "C"
