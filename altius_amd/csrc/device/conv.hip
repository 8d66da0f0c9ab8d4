// Conv2d on NCHW (the reference unfolds the input and calls sgemm per image and group,
// crates/session_interpreter/src/conv2d.rs:26-211).  Three routes:
//
//   depthwise   one input channel per group: 2 k^2 flop per output and no reuse across channels, so the convolution is
//               bound by reading x and writing y once.  conv_depthwise, over tiles in LDS.
//   in place    one product per group, W[oc / group, K] times the unfolded input [K, batch * oh * ow] with
//               K = c / group * kh * kw, whose second operand is read from x in place (an element's address is worked out
//               from its k and its output position; 1 x 1 kernels need no more than k * ih * iw).  The columns of all images
//               are one axis, so that small images fill whole tiles.  conv_gemm_small, which cuts K over the wavefronts of a
//               block, in tiles of 16 x 16 or 32 x 32, or conv_gemm_tiled.
//   unfolded    the general fp32 product (matmul.hip), batched over the images, of the input as it lies (1 x 1 kernels) or of
//               an unfolded copy: its tiles go to LDS without passing registers, k can be cut over blocks, and an element's
//               address is worked out once instead of once per tile of output channels.  Ahead where K and the output
//               channels are many.
//
// Which one of the last two, and which tile, is decided by what each is estimated to take (conv_route).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.h"
#include "ctx.h"
#include "math.h"

namespace altius {
namespace {

using namespace dev;

constexpr int BLOCK = 256;
constexpr size_t MAX_GRID_Y = 65535;
constexpr size_t DW_LDS_FLOATS = 8192;  // 32 KB: five blocks to a CU

// What follows the convolution in the graph (ConvPost), done to a value before it is stored.  A pass of its own over the result costs 2
// to 4 us of launch on one image and 3 to 10 us on 32 of 224 x 224; here it costs 0 to 2 (the stem's square root and division 8).  A
// classifier of that size, 36 convolutions: with the average pool's division and the gates' hard swish in their kernels too 122 launches
// became 73, 662 us 486 on 32 images and 502 365 on one.  The kernels' POST is false where nothing follows: with the code for it in
// them, and nothing to do, they were 5 to 15 % slower (depthwise [59,80,65,65], 1 x 1: 102 and 119 us).
struct Post {
    const float *mean = nullptr, *var = nullptr, *scale = nullptr, *shift = nullptr, *residual = nullptr;
    float eps = 0.0f, alpha = 0.0f, beta = 0.0f;
    int act = 0;
    bool any() const { return mean || act || residual; }
    // ch: output channel, at: where the value goes in the output
    __device__ __forceinline__ float operator()(float v, uint32_t ch, size_t at) const {
        if (mean) v = ((v - mean[ch]) / sqrtf(var[ch] + eps)) * scale[ch] + shift[ch];
        if (act) v = activation(v, act, alpha, beta);
        if (residual) v += residual[at];
        return v;
    }
    // The same for the groups behind the first ones, of `channels` output channels and `floats` of the output's floats.
    Post behind(size_t channels, size_t floats) const {
        Post p = *this;
        if (mean) p.mean += channels, p.var += channels, p.scale += channels, p.shift += channels;
        if (residual) p.residual += floats;
        return p;
    }
};

struct DepthwiseArgs {
    const float *x, *w, *bias;
    float *out;
    FastDiv cols, ygroups;          // decode of an item: output column, group of RY output rows, plane of the block
    FastDiv in_cols, in_rows;       // decode of an LDS tile element
    FastDiv tiles_x, tiles_y;       // decode of the block id: column tile, row tile, group of planes
    FastDiv oc, mult;               // output plane -> channel; output channels per input channel
    uint32_t planes, plane_step;    // output planes in all, and per block
    uint32_t rows;                  // output rows per block (ygroups * RY, rounded up)
    uint32_t c, ih, iw, oh, ow, kh, kw, sh, sw, dh, dw;
    int32_t pad_t, pad_l;
    Post post;
};

// A block owns `plane_step` planes (one, when a plane is cut into tiles) of rows x cols outputs and stages the input they
// read, zero-padded at the borders, in LDS: x comes from memory once (plus the halo between tiles of one plane) and a
// row's k columns are read by neighbouring lanes from consecutive banks.  A thread computes RY outputs of one column, so
// that an input row it has read serves up to K of them: 8 K instead of 4 K^2 LDS reads for K = 5, RY = 4.
// K = 0: any kernel, stride and dilation, RY = 1.  The taps are added in row-major order in every variant.
// [32,240,14,14], 5 x 5: 9.4 us; one product launch per channel took 1.3 ms (240 launches of 5.4 us).
template <int K, int SH, int RY, bool POST>
__global__ __launch_bounds__(BLOCK) void conv_depthwise(DepthwiseArgs g) {
    extern __shared__ float lds[];
    const int tid = threadIdx.x;
    const uint32_t q = g.tiles_x.div(blockIdx.x), tx = blockIdx.x - q * g.tiles_x.d;
    const uint32_t pg = g.tiles_y.div(q), ty = q - pg * g.tiles_y.d;
    const uint32_t plane0 = pg * g.plane_step, n_planes = min(g.plane_step, g.planes - plane0);
    const uint32_t y0 = ty * g.rows, x0 = tx * g.cols.d;
    const uint32_t taps = g.kh * g.kw, tile = g.in_rows.d * g.in_cols.d;
    float *wt = lds + (size_t)g.plane_step * tile;

    for (uint32_t i = tid; i < n_planes * taps; i += BLOCK) {
        const uint32_t p = i / taps, pl = plane0 + p;
        const uint32_t ch = pl - g.oc.div(pl) * g.oc.d;
        wt[i] = g.w[(size_t)ch * taps + (i - p * taps)];
    }
    const int gy0 = (int)(y0 * g.sh) - g.pad_t, gx0 = (int)(x0 * g.sw) - g.pad_l;
    const uint32_t n = n_planes * tile;
    constexpr int BATCH = 4;  // loads in flight per thread
    for (uint32_t base = tid; base < n; base += BLOCK * BATCH) {
        float v[BATCH];
#pragma unroll
        for (int u = 0; u < BATCH; u++) {
            const uint32_t i = base + u * BLOCK;
            v[u] = 0.0f;
            if (i < n) {
                const uint32_t r = g.in_cols.div(i), col = i - r * g.in_cols.d;
                const uint32_t p = g.in_rows.div(r), row = r - p * g.in_rows.d;
                const int yy = gy0 + (int)row, xx = gx0 + (int)col;
                if (yy >= 0 && yy < (int)g.ih && xx >= 0 && xx < (int)g.iw) {
                    const uint32_t pl = plane0 + p, b = g.oc.div(pl), ch = g.mult.div(pl - b * g.oc.d);
                    v[u] = g.x[((size_t)(b * g.c + ch) * g.ih + (uint32_t)yy) * g.iw + (uint32_t)xx];
                }
            }
        }
#pragma unroll
        for (int u = 0; u < BATCH; u++)
            if (base + u * BLOCK < n) lds[base + u * BLOCK] = v[u];
    }
    __syncthreads();

    const uint32_t items = n_planes * g.ygroups.d * g.cols.d;
    for (uint32_t i = tid; i < items; i += BLOCK) {
        const uint32_t r = g.cols.div(i), col = i - r * g.cols.d;
        const uint32_t p = g.ygroups.div(r), yg = r - p * g.ygroups.d;
        const uint32_t x = x0 + col, y = y0 + yg * RY;
        if (x >= g.ow || y >= g.oh) continue;
        const float *t = lds + (size_t)p * tile + (size_t)(yg * RY * g.sh) * g.in_cols.d + col * g.sw;
        const float *wp = wt + p * taps;
        float acc[RY];
#pragma unroll
        for (int o = 0; o < RY; o++) acc[o] = 0.0f;
        if constexpr (K > 0) {
            float w[K * K];
#pragma unroll
            for (int k = 0; k < K * K; k++) w[k] = wp[k];
#pragma unroll
            for (int iy = 0; iy < (RY - 1) * SH + K; iy++) {
                float v[K];
#pragma unroll
                for (int fx = 0; fx < K; fx++) v[fx] = t[iy * g.in_cols.d + fx];
#pragma unroll
                for (int o = 0; o < RY; o++) {
                    const int fy = iy - o * SH;
                    if (fy >= 0 && fy < K) {
#pragma unroll
                        for (int fx = 0; fx < K; fx++) acc[o] = __builtin_fmaf(w[fy * K + fx], v[fx], acc[o]);
                    }
                }
            }
        } else {
            for (uint32_t fy = 0; fy < g.kh; fy++)
                for (uint32_t fx = 0; fx < g.kw; fx++)
                    acc[0] = __builtin_fmaf(wp[fy * g.kw + fx], t[fy * g.dh * g.in_cols.d + fx * g.dw], acc[0]);
        }
        const uint32_t pl = plane0 + p, ch = pl - g.oc.div(pl) * g.oc.d;
        const float bias = g.bias ? g.bias[ch] : 0.0f;
        const size_t at = ((size_t)pl * g.oh + y) * g.ow + x;
#pragma unroll
        for (int k = 0; k < RY; k++)
            if (y + k < g.oh) {
                const float v = g.bias ? acc[k] + bias : acc[k];
                const size_t here = at + (size_t)k * g.ow;
                g.out[here] = POST ? g.post(v, ch, here) : v;
            }
    }
}

// Returns false (nothing launched) for a geometry that products are better for: one whose tile does not fit LDS or whose indices do
// not fit 31 bits, and one whose blocks read far more than they need or have little to compute (rows or columns of the kernel far
// apart, kernels of thousands of taps): a tile of [1,1,2500,2000], 2 x 1 with dilation 2000, holds 8004 values for 4 outputs and
// takes 8.8 ms, against 24 us as a product; [16,256,33,33], 3 x 3, takes 15 us at dilation 1, 77 at 24 (117 as a product) and 216 at
// 36 (110).  Both sides' estimates are fitted to 68 geometries from 3 x 3 to 64 x 64 taps, dilations up to 2000 and strides up to 128.
bool launch_depthwise(DeviceCtx &ctx, float *out, const float *x, const float *w, const float *bias, size_t batch, size_t c, size_t ih,
                      size_t iw, size_t oc, size_t oh, size_t ow, size_t kh, size_t kw, size_t sh, size_t sw, size_t dh, size_t dw,
                      size_t pad_t, size_t pad_l, const Post &post) {
    const size_t lim = (size_t)1 << 31, planes = batch * oc;
    if (planes >= lim || ih >= lim / 4 || iw >= lim / 4 || oh >= lim / 4 || ow >= lim / 4 || kh >= 4096 || kw >= 4096 || sh >= 4096 || sw >= 4096 ||
        dh >= 4096 || dw >= 4096 || pad_t >= lim / 4 || pad_l >= lim / 4 || oh * sh >= lim / 4 || ow * sw >= lim / 4)
        return false;
    const bool square = kh == kw && (kh == 3 || kh == 5) && dh == 1 && dw == 1 && (sh == 1 || sh == 2);
    // Four outputs per thread once that still leaves every CU two blocks; below, one output per thread spreads further.
    const size_t cus = ctx.cus_per_xcd ? (size_t)ctx.cus_per_xcd * 8 : 256;
    const size_t ry = square && planes * ow * ((oh + 3) / 4) >= 2 * cus * BLOCK ? 4 : 1;
    auto up = [](size_t a, size_t b) { return (a + b - 1) / b; };
    size_t tiles_x = up(ow, 64), cols = up(ow, tiles_x);
    size_t ygroups = std::min(up(oh, ry), std::max<size_t>(1, up(BLOCK, cols))), tiles_y = up(up(oh, ry), ygroups);
    ygroups = up(up(oh, ry), tiles_y);
    size_t step = tiles_x == 1 && tiles_y == 1 ? std::max<size_t>(1, BLOCK / (cols * ygroups)) : 1;
    auto in_rows = [&] { return (ygroups * ry - 1) * sh + (kh - 1) * dh + 1; };
    auto in_cols = [&] { return (cols - 1) * sw + (kw - 1) * dw + 1; };
    auto floats = [&] { return step * (in_rows() * in_cols() + kh * kw); };
    while (floats() > DW_LDS_FLOATS) {
        if (step > 1) step /= 2;
        else if (ygroups > 1) tiles_y = up(up(oh, ry), ygroups = (ygroups + 1) / 2);
        else if (cols > 1) tiles_x = up(ow, cols = (cols + 1) / 2);
        else return false;
    }
    step = std::min(step, planes);
    const size_t blocks = tiles_x * tiles_y * up(planes, step);
    if (blocks * BLOCK > 0xffffffffu) return false;  // a grid ends at 2^32 threads
    const double tap_rounds = square ? 0.0 : (double)(kh * kw * up(step * ygroups * cols, BLOCK));
    const double here_us = 3.0 + 0.03 * tap_rounds + (double)blocks * (6e-4 + 6.7e-7 * (double)floats() + 2.6e-5 * tap_rounds);
    const size_t chunks = up(kh * kw, 16);
    const double product_us = 3.0 + 0.5 * (double)up(chunks, 8) + 3.6e-4 * (double)(up(oc / c, 16) * up(batch * oh * ow, 16) * c * chunks);
    if (here_us > 1.25 * product_us) return false;
    DepthwiseArgs g;
    g.x = x, g.w = w, g.bias = bias, g.out = out;
    g.cols = make_fastdiv((uint32_t)cols), g.ygroups = make_fastdiv((uint32_t)ygroups);
    g.in_cols = make_fastdiv((uint32_t)in_cols()), g.in_rows = make_fastdiv((uint32_t)in_rows());
    g.tiles_x = make_fastdiv((uint32_t)tiles_x), g.tiles_y = make_fastdiv((uint32_t)tiles_y);
    g.oc = make_fastdiv((uint32_t)oc), g.mult = make_fastdiv((uint32_t)(oc / c));
    g.planes = (uint32_t)planes, g.plane_step = (uint32_t)step, g.rows = (uint32_t)(ygroups * ry);
    g.c = (uint32_t)c, g.ih = (uint32_t)ih, g.iw = (uint32_t)iw, g.oh = (uint32_t)oh, g.ow = (uint32_t)ow;
    g.kh = (uint32_t)kh, g.kw = (uint32_t)kw, g.sh = (uint32_t)sh, g.sw = (uint32_t)sw, g.dh = (uint32_t)dh, g.dw = (uint32_t)dw;
    g.pad_t = (int32_t)pad_t, g.pad_l = (int32_t)pad_l;
    g.post = post;
    const dim3 grid((unsigned)blocks);
    const size_t lds = floats() * sizeof(float);
#define DEPTHWISE(K, SH, RY)                                                                                                      \
    do {                                                                                                                           \
        if (post.any()) hipLaunchKernelGGL((conv_depthwise<K, SH, RY, true>), grid, dim3(BLOCK), lds, ctx.stream, g);              \
        else hipLaunchKernelGGL((conv_depthwise<K, SH, RY, false>), grid, dim3(BLOCK), lds, ctx.stream, g);                        \
    } while (0)
    if (!square) DEPTHWISE(0, 1, 1);
    else if (ry == 1 && kh == 3) DEPTHWISE(3, 1, 1);
    else if (ry == 1) DEPTHWISE(5, 1, 1);
    else if (kh == 3 && sh == 1) DEPTHWISE(3, 1, 4);
    else if (kh == 3) DEPTHWISE(3, 2, 4);
    else if (sh == 1) DEPTHWISE(5, 1, 4);
    else DEPTHWISE(5, 2, 4);
#undef DEPTHWISE
    return true;
}


// ---- products over the unfolded input ------------------------------------------------------------------------------

typedef float floatx4 __attribute__((ext_vector_type(4)));

struct ConvGemmArgs {
    const float *x, *w, *bias;
    float *out;
    FastDiv ohw, ow;       // column -> image, row, column of the output
    FastDiv taps, kw;      // k -> input channel, row and column of the kernel
    uint32_t m, n, k;      // output channels per group, columns of all images, c / group * kh * kw
    uint32_t c, cg, oc, ih, iw, sh, sw, dh, dw;
    int32_t pad_t, pad_l;
    uint32_t tiles_n;
    int w_vec, x_vec;      // 16-byte loads along k of w; along a row of x (1 x 1 kernels)
    Post post;
};

// Where one column of the unfolded input starts in x, for the group whose first channel `x` points at.
template <bool POINTWISE> struct Column {
    const float *p;  // channel 0 of the column's image (POINTWISE: at the column's own position)
    int y, x;        // the kernel's top left corner in the image
    __device__ __forceinline__ Column(const ConvGemmArgs &g, const float *xg, uint32_t n) {
        const uint32_t b = g.ohw.div(n), pos = n - b * g.ohw.d;
        p = xg + (size_t)b * g.c * g.ih * g.iw;
        if (POINTWISE) {
            p += pos;
            y = x = 0;
        } else {
            const uint32_t oy = g.ow.div(pos), ox = pos - oy * g.ow.d;
            y = (int)(oy * g.sh) - g.pad_t;
            x = (int)(ox * g.sw) - g.pad_l;
        }
    }
    // k < g.k
    __device__ __forceinline__ float at(const ConvGemmArgs &g, uint32_t k) const {
        if (POINTWISE) return p[(size_t)k * g.ohw.d];
        const uint32_t ch = g.taps.div(k), t = k - ch * g.taps.d, fy = g.kw.div(t), fx = t - fy * g.kw.d;
        const int yy = y + (int)(fy * g.dh), xx = x + (int)(fx * g.dw);
        if (yy < 0 || yy >= (int)g.ih || xx < 0 || xx >= (int)g.iw) return 0.0f;
        return p[((size_t)ch * g.ih + (uint32_t)yy) * g.iw + (uint32_t)xx];
    }
};

__device__ __forceinline__ size_t out_offset(const ConvGemmArgs &g, uint32_t channel, uint32_t n) {
    const uint32_t b = g.ohw.div(n), pos = n - b * g.ohw.d;
    return ((size_t)b * g.oc + channel) * g.ohw.d + pos;
}

// Four consecutive k of one row of w from k0 on, zeros past the end.
__device__ __forceinline__ floatx4 weights4(const float *row, uint32_t k0, uint32_t k, int vec) {
    if (vec && k0 + 3 < k) return *reinterpret_cast<const floatx4 *>(row + k0);
    floatx4 v = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < 4; j++)
        if (k0 + j < k) v[j] = row[k0 + j];
    return v;
}

// One block per 16 MT x 16 NT tile; its wavefronts take every 16 th chunk of k in turn, straight from memory (nothing is
// shared between them, so nothing goes through LDS but the final sum, in wavefront order).  With the small products of one
// image the whole time is the latency of one chain of loads; cutting k shortens the chain and brings more of them into
// flight: 96 x 49 over k = 576 takes 3.8 us, against 3.0 for an im2col and 5 to 10 for the general product of its result.
// (Requesting the next chunk ahead of the products was measured: equal for one tile, 9.1 -> 11.5 us for 2 x 2.)
// The k of an MFMA may be any four as long as both operands agree: lane q of four takes k0 + 4 q + j in step j, so that
// a lane's share of w is one 16-byte load per four steps.
template <bool POINTWISE, int MT, int NT, bool POST>
__global__ __launch_bounds__(512) void conv_gemm_small(ConvGemmArgs g) {
    extern __shared__ float lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
    const uint32_t tm = blockIdx.x / g.tiles_n, tn = blockIdx.x - tm * g.tiles_n, grp = blockIdx.y;
    const float *xg = g.x + (size_t)grp * g.cg * g.ih * g.iw, *wg = g.w + (size_t)grp * g.m * g.k;
    const int r = lane & 15, q = lane >> 4;
    const float *row[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) row[i] = wg + (size_t)min(tm * (16 * MT) + i * 16 + r, g.m - 1) * g.k;
    const Column<POINTWISE> c0(g, xg, min(tn * (16 * NT) + r, g.n - 1)), c1(g, xg, min(tn * (16 * NT) + 16 * (NT - 1) + r, g.n - 1));

    floatx4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t chunk = wave * 16; chunk < g.k; chunk += waves * 16) {
        const uint32_t k0 = chunk + q * 4;
        floatx4 a[MT];
        float b[NT][4];
#pragma unroll
        for (int i = 0; i < MT; i++) a[i] = weights4(row[i], k0, g.k, g.w_vec);
#pragma unroll
        for (int s = 0; s < 4; s++) {
            b[0][s] = k0 + s < g.k ? c0.at(g, k0 + s) : 0.0f;
            if (NT > 1) b[NT - 1][s] = k0 + s < g.k ? c1.at(g, k0 + s) : 0.0f;
        }
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][s], b[j][s], acc[i][j], 0, 0, 0);
    }
    // Accumulator e of lane l is row 4 * (l / 16) + e, column l % 16 of its 16 x 16 tile.
    constexpr int TILE = 256 * MT * NT, WIDTH = 16 * NT;
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) lds[wave * TILE + (i * 16 + q * 4 + e) * WIDTH + j * 16 + r] = acc[i][j][e];
    __syncthreads();
    for (int i = tid; i < TILE; i += blockDim.x) {
        float v = lds[i];
        for (int u = 1; u < waves; u++) v += lds[u * TILE + i];
        const uint32_t mm = tm * (16 * MT) + i / WIDTH, n = tn * WIDTH + i % WIDTH;
        if (mm >= g.m || n >= g.n) continue;
        const uint32_t ch = grp * g.m + mm;
        if (g.bias) v += g.bias[ch];
        const size_t at = out_offset(g, ch, n);
        g.out[at] = POST ? g.post(v, ch, at) : v;
    }
}

// 64 x 128 tile per block of four wavefronts (32 x 64 each), k in steps of 16 through two LDS buffers; the loads of step
// t + 1 are in flight during the products of step t.  [72,16] x [16, 32 * 3136] takes 15 us here.  w lies in LDS as [row][k]
// (pitch 20: the 16-byte reads of 16 rows meet all 64 banks), x as [k][column] (pitch 132: the four k of a step are 16 banks apart).
constexpr int TM = 64, TN = 128, TK = 16, WP = TK + 4, XP = TN + 4;

template <bool POINTWISE, bool POST>
__global__ __launch_bounds__(BLOCK) void conv_gemm_tiled(ConvGemmArgs g) {
    __shared__ __align__(16) float ws[2][TM * WP];
    __shared__ __align__(16) float xs[2][TK * XP];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, q = lane >> 4;
    const uint32_t tm = blockIdx.x / g.tiles_n, tn = blockIdx.x - tm * g.tiles_n, grp = blockIdx.y;
    const float *xg = g.x + (size_t)grp * g.cg * g.ih * g.iw, *wg = g.w + (size_t)grp * g.m * g.k;
    const uint32_t m0 = tm * TM, n0 = tn * TN;
    const int wm = wave >> 1, wn = wave & 1;

    // w: row tid / 4, four k from 4 * (tid % 4) on.  x, 16 bytes at a time: k = tid / 32 and + 8, columns 4 * (tid % 32) on;
    // one value at a time: column tid % 128, k = tid / 128 + 2 u.
    const float *wrow = wg + (size_t)min(m0 + (tid >> 2), g.m - 1) * g.k;
    const bool vec = POINTWISE && g.x_vec;
    const Column<POINTWISE> col(g, xg, vec ? min(n0 + (tid & 31) * 4, (g.n - 1) & ~3u) : min(n0 + (tid & 127), g.n - 1));
    floatx4 wr;
    float xr[8];
    auto load = [&](uint32_t k0) {
        wr = weights4(wrow, k0 + (tid & 3) * 4, g.k, g.w_vec);
        if (vec) {
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const uint32_t k = k0 + (tid >> 5) + 8 * u;
                floatx4 v = {0.0f, 0.0f, 0.0f, 0.0f};
                if (k < g.k) v = *reinterpret_cast<const floatx4 *>(col.p + (size_t)k * g.ohw.d);
#pragma unroll
                for (int e = 0; e < 4; e++) xr[4 * u + e] = v[e];
            }
        } else {
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const uint32_t k = k0 + (tid >> 7) + 2 * u;
                xr[u] = k < g.k ? col.at(g, k) : 0.0f;
            }
        }
    };
    auto store = [&](int buf) {
        *reinterpret_cast<floatx4 *>(&ws[buf][(tid >> 2) * WP + (tid & 3) * 4]) = wr;
        if (vec) {
#pragma unroll
            for (int u = 0; u < 2; u++)
                *reinterpret_cast<floatx4 *>(&xs[buf][((tid >> 5) + 8 * u) * XP + (tid & 31) * 4]) = floatx4{xr[4 * u], xr[4 * u + 1], xr[4 * u + 2], xr[4 * u + 3]};
        } else {
#pragma unroll
            for (int u = 0; u < 8; u++) xs[buf][((tid >> 7) + 2 * u) * XP + (tid & 127)] = xr[u];
        }
    };
    floatx4 acc[2][4];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    load(0);
    store(0);
    __syncthreads();
    const uint32_t steps = (g.k + TK - 1) / TK;
    for (uint32_t t = 0; t < steps; t++) {
        const int cur = t & 1;
        if (t + 1 < steps) load((t + 1) * TK);
        floatx4 a[2];
#pragma unroll
        for (int i = 0; i < 2; i++) a[i] = *reinterpret_cast<const floatx4 *>(&ws[cur][(wm * 32 + i * 16 + r) * WP + q * 4]);
#pragma unroll
        for (int s = 0; s < 4; s++) {
            float b[4];
#pragma unroll
            for (int j = 0; j < 4; j++) b[j] = xs[cur][(q * 4 + s) * XP + wn * 64 + j * 16 + r];
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][s], b[j], acc[i][j], 0, 0, 0);
        }
        if (t + 1 < steps) store(cur ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t n = n0 + wn * 64 + j * 16 + r;
        if (n >= g.n) continue;
        const size_t first = out_offset(g, grp * g.m, n);
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t mm = m0 + wm * 32 + i * 16 + q * 4 + e;
                if (mm >= g.m) continue;
                const uint32_t ch = grp * g.m + mm;
                const size_t at = first + (size_t)mm * g.ohw.d;
                const float v = g.bias ? acc[i][j][e] + g.bias[ch] : acc[i][j][e];
                g.out[at] = POST ? g.post(v, ch, at) : v;
            }
    }
}

// col[image][c][fy][fx][oh][ow] = x[image][c][oh * sh - pad_t + fy * dh][ow * sw - pad_l + fx * dw], zero outside the image
// (conv2d.rs:82-150, 213-333).  Bound by writing col: 2.0 us per million elements.
struct UnfoldArgs {
    FastDiv ow, oh, kw, kh;
    uint32_t ih, iw, sh, sw, dh, dw, total;
    int32_t pad_t, pad_l;
};

__global__ __launch_bounds__(BLOCK) void conv_unfold(float *__restrict__ col, const float *__restrict__ x, UnfoldArgs g) {
    const uint32_t i = blockIdx.x * BLOCK + threadIdx.x;
    if (i >= g.total) return;
    const uint32_t r1 = g.ow.div(i), ox = i - r1 * g.ow.d;
    const uint32_t r2 = g.oh.div(r1), oy = r1 - r2 * g.oh.d;
    const uint32_t r3 = g.kw.div(r2), fx = r2 - r3 * g.kw.d;
    const uint32_t plane = g.kh.div(r3), fy = r3 - plane * g.kh.d;
    const int yy = (int)(oy * g.sh + fy * g.dh) - g.pad_t, xx = (int)(ox * g.sw + fx * g.dw) - g.pad_l;
    float v = 0.0f;
    if (yy >= 0 && yy < (int)g.ih && xx >= 0 && xx < (int)g.iw) v = x[((size_t)plane * g.ih + (uint32_t)yy) * g.iw + (uint32_t)xx];
    col[i] = v;
}

// The unfolded copy lives in the context's workspace, of as many images at a time as this holds, or of as many output rows of one
// image: 1 GiB ([32,2048,28,28] -> 256, 3 x 3: 4010 us in passes of four images, 256 MiB; 3570 in two passes).
constexpr size_t UNFOLD_FLOATS = (size_t)256 << 20;

enum Route { SMALL_16, SMALL_32, TILED, UNFOLDED };

// What a launch of an in-place kernel takes, in us, over `chunks` of 16 values of k: base + chain * (chunks one wavefront walks)
// + tiles * (chunk * chunks + tile) for the small ones; for the tiled one rounds * (tile + chunk * chunks), of 256 tiles each, or
// alone + alone_chunk * chunks where that is one.  The unfolded route takes its own kernel and one product per group.  Fitted to 336
// geometries (1 x 1 to 16 x 16 taps, 3 to 2048 channels, images of 7 x 7 to 224 x 224, batches of 1 to 64, up to 32 groups), every
// route timed on each: within 9 % (rms) of the unfolded one, 9 to 15 % of the tiled and 16 to 24 % of the small ones, and the route
// chosen is 1.5 % behind the best one on average.  (Before, tiles from 512 of them on and no unfolded route: 19 %;
// [32,1024,14,14] -> 2048, 1 x 1 with stride 2: 260 us, 95 unfolded; [4,320,64,64] -> 320, 3 x 3: 555 and 322.)
struct SmallCost { double base, chain, chunk, tile; };
struct TiledCost { double base, tile, chunk, alone, alone_chunk; };
constexpr SmallCost SMALL_COST[2][2] = {{{2.8, 0.55, 0.28e-3, 0.41e-3}, {2.8, 0.11, 0.27e-3, 0.16e-3}},   // 16 x 16: windows, pointwise
                                        {{2.9, 1.26, 0.65e-3, 1.10e-3}, {2.9, 0.68, 0.62e-3, 0.66e-3}}};  // 32 x 32
constexpr TiledCost TILED_COST[2] = {{6.0, 0.5, 1.01, 0.0, 1.82}, {3.6, 1.75, 0.64, 3.4, 0.94}};

// What the unfolded route takes at a time: `images` images, or `rows` output rows of one; none where it cannot be taken.
struct Pass { size_t images = 0, rows = 0; };

Route conv_route(const DeviceCtx &ctx, size_t batch, size_t m, size_t oh, size_t ow, size_t k, size_t group, Pass pass, bool pointwise, bool vec) {
    auto up = [](size_t a, size_t b) { return (a + b - 1) / b; };
    const size_t n = batch * oh * ow, chunks = up(k, 16), waves = std::min<size_t>(8, std::max<size_t>(1, chunks));
    const TiledCost &t = TILED_COST[pointwise];
    const size_t rounds = up(up(m, TM) * up(n, TN) * group, 256);
    Route best = TILED;
    double best_us = t.base + (rounds > 1 ? (double)rounds * (t.tile + t.chunk * (double)chunks) : t.alone + t.alone_chunk * (double)chunks);
    for (size_t s = 0; s < 2; s++) {
        const size_t tiles = up(m, 16 << s) * up(n, 16 << s);
        if (tiles * 64 * waves > 0xffffffffu) continue;  // a grid ends at 2^32 threads
        const SmallCost &c = SMALL_COST[s][pointwise];
        const double us = c.base + c.chain * (double)up(chunks, waves) + (double)(tiles * group) * (c.chunk * (double)chunks + c.tile);
        if (us < best_us) best_us = us, best = s ? SMALL_32 : SMALL_16;
    }
    if (pass.images) {
        const size_t cols = pass.rows * ow;
        const double pass_us = (pointwise ? 0.0 : 2.8 + 2.0e-6 * (double)(pass.images * group * k * cols)) +
                               (double)group * gemm_f32_us(ctx, pass.images, m, cols, k, vec);
        if ((double)(batch * oh) / (double)(pass.images * pass.rows) * pass_us < best_us) best = UNFOLDED;
    }
    return best;
}

int launch_unfolded(DeviceCtx &ctx, float *out, const float *x, const float *w, const float *bias, Pass pass, bool pointwise, size_t batch, size_t c,
                    size_t ih, size_t iw, size_t oc, size_t oh, size_t ow, size_t kh, size_t kw, size_t sh, size_t sw, size_t dh, size_t dw, size_t pad_t,
                    size_t pad_l, size_t group, const GemmPost &then) {
    const size_t ohw = oh * ow, m = oc / group, k = c / group * kh * kw;
    void *ws = nullptr;
    if (!pointwise)
        if (int rc = gemm_workspace(ctx, pass.images * c * kh * kw * pass.rows * ow * sizeof(float), &ws)) return rc;
    for (size_t b0 = 0; b0 < batch; b0 += pass.images)
        for (size_t y0 = 0; y0 < oh; y0 += pass.rows) {
            const size_t images = std::min(pass.images, batch - b0), rows = std::min(pass.rows, oh - y0), cols = rows * ow, total = images * c * kh * kw * cols;
            const float *src = x + b0 * c * ih * iw;
            if (!pointwise) {
                UnfoldArgs g;
                g.ow = make_fastdiv((uint32_t)ow), g.oh = make_fastdiv((uint32_t)rows), g.kw = make_fastdiv((uint32_t)kw), g.kh = make_fastdiv((uint32_t)kh);
                g.ih = (uint32_t)ih, g.iw = (uint32_t)iw, g.sh = (uint32_t)sh, g.sw = (uint32_t)sw, g.dh = (uint32_t)dh, g.dw = (uint32_t)dw;
                g.pad_t = (int32_t)((int64_t)pad_t - (int64_t)(y0 * sh)), g.pad_l = (int32_t)pad_l, g.total = (uint32_t)total;
                hipLaunchKernelGGL(conv_unfold, dim3((unsigned)((total + BLOCK - 1) / BLOCK)), dim3(BLOCK), 0, ctx.stream, static_cast<float *>(ws), src, g);
                if (int rc = ctx.check(hipGetLastError(), "conv2d launch")) return rc;
                src = static_cast<const float *>(ws);
            }
            const size_t none[2] = {0, 0}, b_bs[2] = {group * k * cols, 0}, c_bs[2] = {oc * ohw, 0};
            for (size_t q = 0; q < group; q++) {
                const size_t at = (b0 * oc + q * m) * ohw + y0 * ow;
                GemmPost post = then;
                if (post.residual) post.residual += at;
                const int rc = launch_gemm_f32(ctx, out + at, w + q * m * k, src + q * k * cols, bias ? bias + q * m : nullptr,
                                               images, 1, m, cols, k, 0, 0, k, cols, ohw, none, b_bs, c_bs, 1, 0, 1.0f, bias ? 1.0f : 0.0f, &post);
                if (rc) return rc;
            }
        }
    return AHIP_OK;
}

}  // namespace

int launch_conv2d(DeviceCtx &ctx, float *out, const float *x, const float *w, const float *bias, size_t batch, size_t c, size_t ih, size_t iw,
                  size_t oc, size_t oh, size_t ow, size_t kh, size_t kw, size_t sh, size_t sw, size_t dh, size_t dw, size_t pad_t, size_t pad_l,
                  size_t group, ConvPost *conv_post) {
    if (conv_post) conv_post->applied = false;
    if (batch == 0 || oc == 0 || oh == 0 || ow == 0) return AHIP_OK;
    if (group == 0 || c % group || oc % group) return ctx.fail(AHIP_ERR_SHAPE, "conv2d: channels do not divide into the groups");
    if (!out || !x || !w) return ctx.fail(AHIP_ERR_ARG, "conv2d: null pointer");
    Post post;
    if (conv_post) {
        const GemmPost &t = conv_post->then;
        post.mean = conv_post->mean, post.var = conv_post->var, post.scale = conv_post->scale, post.shift = conv_post->shift, post.eps = conv_post->eps;
        post.act = t.act, post.alpha = t.alpha, post.beta = t.beta, post.residual = t.residual;
    }
    auto launched = [&] {
        if (conv_post) conv_post->applied = true;
        return ctx.check(hipGetLastError(), "conv2d launch");
    };
    if (group == c && launch_depthwise(ctx, out, x, w, bias, batch, c, ih, iw, oc, oh, ow, kh, kw, sh, sw, dh, dw, pad_t, pad_l, post)) return launched();
    const size_t lim = (size_t)1 << 31, cg = c / group, m = oc / group, k = cg * kh * kw, n = batch * oh * ow;
    if (n >= lim || k >= lim || m >= lim || c >= lim || oc >= lim || ih >= lim || iw >= lim || (oh - 1) * sh + pad_t >= lim ||
        (ow - 1) * sw + pad_l >= lim || (oh - 1) * sh + (kh - 1) * dh >= lim || (ow - 1) * sw + (kw - 1) * dw >= lim)
        return ctx.fail(AHIP_ERR_UNSUPPORTED, "conv2d: extent above 2^31");
    ConvGemmArgs g;
    g.ohw = make_fastdiv((uint32_t)(oh * ow)), g.ow = make_fastdiv((uint32_t)ow);
    g.taps = make_fastdiv((uint32_t)(kh * kw)), g.kw = make_fastdiv((uint32_t)kw);
    g.m = (uint32_t)m, g.n = (uint32_t)n, g.k = (uint32_t)k;
    g.c = (uint32_t)c, g.cg = (uint32_t)cg, g.oc = (uint32_t)oc, g.ih = (uint32_t)ih, g.iw = (uint32_t)iw;
    g.sh = (uint32_t)sh, g.sw = (uint32_t)sw, g.dh = (uint32_t)dh, g.dw = (uint32_t)dw;
    g.pad_t = (int32_t)pad_t, g.pad_l = (int32_t)pad_l;
    const bool pointwise = kh == 1 && kw == 1 && sh == 1 && sw == 1 && pad_t == 0 && pad_l == 0 && ih == oh && iw == ow;
    auto a16 = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    g.w_vec = k % 4 == 0 && a16(w);
    g.x_vec = pointwise && (ih * iw) % 4 == 0 && a16(x);
    auto up = [](size_t a, size_t b) { return (a + b - 1) / b; };
    auto grid = [&](size_t bm, size_t bn) {
        g.tiles_n = (uint32_t)up(n, bn);
        return up(m, bm) * up(n, bn);
    };
    Pass pass;
    const size_t row = c * kh * kw * ow;  // floats of one output row, unfolded; the product's rows of 2^24 columns are far apart (matmul.hip)
    if (pointwise) pass.images = batch, pass.rows = oh;
    else if (row && row * oh <= UNFOLD_FLOATS) pass.images = up(batch, up(batch, UNFOLD_FLOATS / (row * oh))), pass.rows = oh;
    else if (row && row <= UNFOLD_FLOATS) pass.images = 1, pass.rows = up(oh, up(oh, UNFOLD_FLOATS / row));
    if (pass.rows * ow > (size_t)1 << 24) pass.images = 0;
    Route route = conv_route(ctx, batch, m, oh, ow, k, group, pass, pointwise, g.w_vec && (pass.rows * ow) % 4 == 0 && (!pointwise || a16(x)));
    if (route == UNFOLDED) {
        // Without a bias the products of many small images are one launch of matmul_small.hip's kernel, which has no epilogue and adds up in
        // another order than the tiles that have one: what stands behind such a convolution stays with its own node.  (Where images are taken
        // in passes, the first pass has the most of them.)
        const bool takes_post = conv_post && !post.mean && (bias || !gemm_small_batched_fits(pass.images, m, pass.rows * ow, k));
        const int rc = launch_unfolded(ctx, out, x, w, bias, pass, pointwise, batch, c, ih, iw, oc, oh, ow, kh, kw, sh, sw, dh, dw, pad_t, pad_l, group,
                                       takes_post ? conv_post->then : GemmPost());
        if (!rc && conv_post) conv_post->applied = takes_post;
        if (rc != AHIP_ERR_OOM && rc != AHIP_ERR_UNSUPPORTED) return rc;
        route = conv_route(ctx, batch, m, oh, ow, k, group, Pass(), pointwise, false);  // no room for the copy
    }
    const bool tiled = route == TILED, wide = route == SMALL_32;
    const size_t blocks = tiled ? grid(TM, TN) : wide ? grid(32, 32) : grid(16, 16);
    const size_t waves = std::min<size_t>(8, std::max<size_t>(1, up(k, 16))), lds = waves * (wide ? 1024 : 256) * sizeof(float);
    const dim3 block((unsigned)(tiled ? BLOCK : 64 * waves));
    if (blocks * block.x > 0xffffffffu) return ctx.fail(AHIP_ERR_UNSUPPORTED, "conv2d: more tiles than a grid holds");
    // Groups lie along the grid's second axis, which ends at 65535.
    for (size_t g0 = 0; g0 < group; g0 += MAX_GRID_Y) {
        const dim3 dim((unsigned)blocks, (unsigned)std::min(group - g0, MAX_GRID_Y));
        g.x = x + g0 * cg * ih * iw, g.w = w + g0 * m * k, g.bias = bias ? bias + g0 * m : nullptr, g.out = out + g0 * m * oh * ow;
        g.post = post.behind(g0 * m, g0 * m * oh * ow);
#define PRODUCT(KERNEL, ...)                                                                                        \
    do {                                                                                                             \
        if (post.any()) hipLaunchKernelGGL((KERNEL<__VA_ARGS__, true>), dim, block, tiled ? 0 : lds, ctx.stream, g); \
        else hipLaunchKernelGGL((KERNEL<__VA_ARGS__, false>), dim, block, tiled ? 0 : lds, ctx.stream, g);           \
    } while (0)
        if (tiled && pointwise) PRODUCT(conv_gemm_tiled, true);
        else if (tiled) PRODUCT(conv_gemm_tiled, false);
        else if (pointwise && wide) PRODUCT(conv_gemm_small, true, 2, 2);
        else if (pointwise) PRODUCT(conv_gemm_small, true, 1, 1);
        else if (wide) PRODUCT(conv_gemm_small, false, 2, 2);
        else PRODUCT(conv_gemm_small, false, 1, 1);
#undef PRODUCT
    }
    return launched();
}

}  // namespace altius
