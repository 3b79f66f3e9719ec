// unet.hip -- the learned initial guess of the p' solve: a 4-level U-Net
// (16-32-64-128 channels, 3x3 convolutions) with BF16 weights and
// activations and FP32 accumulation on the gfx950 matrix cores
// (v_mfma_f32_16x16x32_bf16), for inference and for training.  No reference
// counterpart: the reference always starts MSI from the caller's var.
//
// Tensors are NHWC (channels fastest), bf16, channel counts multiples of 8,
// so one lane moves 8 channels (16 bytes) at a time.  A convolution is an
// implicit GEMM: M = pixels, N = output channels, K = 9 taps x input
// channels, k = tap * Cin + ci (tap = 3 ky + kx); weights are stored
// [Cout_pad][Kpad] (Kpad = 9 Cin rounded up to 32, zeros beyond).  Its input
// is up to two tensors whose channels are concatenated: the first may be read
// directly, as the 2x2 average of a tensor of twice the resolution (the
// down path's pooling, fused), or as the nearest-neighbour 2x upsampling of a
// tensor of half the resolution (the up path, fused); the second (the skip
// connection) is read directly.  The backward pass reuses the same kernel for
// input gradients (weights rotated by 180 degrees, channels transposed) and
// has its own MFMA kernel for weight gradients.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <type_traits>

#include "m2d_internal.h"
#include "msi_stencil.h"

namespace m2d {
namespace unet {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

constexpr int kMode0 = 0;     // direct
constexpr int kModePool = 1;  // 2x2 average of a 2H x 2W tensor
constexpr int kModeUp = 2;    // nearest 2x upsampling of an H/2 x W/2 tensor

struct In {
    const __bf16 *x;
    int c, mode;
};

struct ConvArgs {
    In in1, in2;          // in2.c == 0: no second input
    const __bf16 *w;      // [cout_pad][kpad]
    const float *bias;    // cout values, or null
    __bf16 *out;          // NHWC, cout_stride channels, or null
    float *out32;         // NHWC fp32, cout_stride channels, or null
    int cout, cout_stride, kpad;
    int n, h, w_;         // output (and direct-input) resolution
    int relu;
    int accumulate;       // add into out32 instead of overwriting
    int vec;              // outputs can be stored four channels at a time
    int tiles_x, tiles_y; // k_conv3x3_tile's tiles of one image
    unsigned rc8, rc1, rc2;  // div_recip(channels / 8): both inputs', each one's
};

__device__ __forceinline__ bf16x8 zero8()
{
    bf16x8 z;
#pragma unroll
    for (int i = 0; i < 8; ++i) z[i] = (__bf16)0.0f;
    return z;
}

__device__ __forceinline__ bf16x8 ld8(const __bf16 *p)
{
    return *reinterpret_cast<const bf16x8 *>(p);
}

// 8 channels ci0.. of the (virtual) input at pixel (n, y, x) of the output
// resolution h x w, for input `in` (tensor resolution per its mode).
__device__ __forceinline__ bf16x8 load_in(const In &in, int ci0, int n, int y, int x, int h,
                                          int w)
{
    if (in.mode == kMode0) return ld8(in.x + (((long)n * h + y) * w + x) * in.c + ci0);
    if (in.mode == kModeUp) {
        const int hc = h >> 1, wc = w >> 1;
        return ld8(in.x + (((long)n * hc + (y >> 1)) * wc + (x >> 1)) * in.c + ci0);
    }
    const int hf = h << 1, wf = w << 1;  // pooled: mean of the 2x2 block
    const __bf16 *p = in.x + (((long)n * hf + 2 * y) * wf + 2 * x) * in.c + ci0;
    const bf16x8 a = ld8(p), b = ld8(p + in.c), c = ld8(p + (long)wf * in.c),
                 d = ld8(p + (long)wf * in.c + in.c);
    bf16x8 r;
#pragma unroll
    for (int i = 0; i < 8; ++i)
        r[i] = (__bf16)((((float)a[i] + (float)b[i]) + ((float)c[i] + (float)d[i])) * 0.25f);
    return r;
}

// im2col element group: 8 consecutive k = k0.. (k0 multiple of 8) of pixel
// p (flat n*h*w index); zeros outside the image and beyond 9 * cin.
__device__ __forceinline__ bf16x8 im2col8(const ConvArgs &A, int p, int k0)
{
    const int cin = A.in1.c + A.in2.c;
    if (k0 >= 9 * cin) return zero8();
    const int tap = k0 / cin, ci0 = k0 - tap * cin;
    const int hw = A.h * A.w_;
    const int n = p / hw, rem = p - n * hw, y0 = rem / A.w_, x0 = rem - y0 * A.w_;
    const int y = y0 + tap / 3 - 1, x = x0 + tap % 3 - 1;
    if (y < 0 || y >= A.h || x < 0 || x >= A.w_) return zero8();
    return ci0 < A.in1.c ? load_in(A.in1, ci0, n, y, x, A.h, A.w_)
                         : load_in(A.in2, ci0 - A.in1.c, n, y, x, A.h, A.w_);
}

// Forward convolution (also the input gradient, with rotated weights) of any
// number of input channels: for those whose staged tile does not fit
// k_conv3x3_tile's LDS.
// Workgroup: 4 waves x 16 pixels; wave: 16 pixels x 16*NT output channels.
template <int NT>
__global__ __launch_bounds__(256) void k_conv3x3(ConvArgs A)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int npix = A.n * A.h * A.w_;
    const int pix0 = (blockIdx.x * 4 + wave) * 16;
    const int co0 = blockIdx.y * 16 * NT;
    if (pix0 >= npix) return;
    const int pa = min(pix0 + (lane & 15), npix - 1);  // A row of this lane
    const int kl = 8 * (lane >> 4);                    // k offset of this lane
    f32x4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    const __bf16 *wrow = A.w + (long)(co0 + (lane & 15)) * A.kpad + kl;
    for (int kb = 0; kb < A.kpad; kb += 32) {
        const bf16x8 a = im2col8(A, pa, kb + kl);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const bf16x8 b = ld8(wrow + (long)t * 16 * A.kpad + kb);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[t], 0, 0, 0);
        }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int co = co0 + 16 * t + (lane & 15);
        if (co >= A.cout) continue;
        const float bias = A.bias ? A.bias[co] : 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int p = pix0 + 4 * (lane >> 4) + i;
            if (p >= npix) continue;
            float v = acc[t][i] + bias;
            if (A.relu) v = fmaxf(v, 0.0f);
            const long o = (long)p * A.cout_stride + co;
            if (A.out) A.out[o] = (__bf16)v;
            if (A.out32) A.out32[o] = A.accumulate ? A.out32[o] + v : v;
        }
    }
}

// Forward convolution through LDS.  A workgroup computes TH = MT WP rows of
// 16 pixels x 16 NT WC output channels: it stages the (TH + 2) x 18 pixels of
// input it needs once (pooling or upsampling them on the way, so a pooled
// value is formed once and not for each of its nine taps) and its waves, WP
// along the rows and WC along the channels, read the taps from there.  The
// weights are the first operand, so a lane ends up with four neighbouring
// channels of one pixel and stores them at once.  Products are added in the
// order of k_conv3x3 (32 k at a time), so both give the same bits.
//   bound: the 16-channel layers of the full resolution by memory (1026x514:
// 45.1 MB in 13.6 us, 3.3 TB/s); the others by latency, of the staged tile, of
// the weights and, in the deep layers, of few workgroups: no unit is near its
// rate (counted over the guess: matrix cores busy for 4 to 13 % of a kernel's
// time, LDS for 4 to 25 %).  A pixel's channels lie an odd number of 16-byte
// units apart, so that 16 neighbouring pixels start in different banks; about
// 46 % of the LDS's busy cycles are conflicts all the same (6 % with 8
// channels).
constexpr int kTileW = 16, kHaloW = kTileW + 2;

// channels between two pixels of the staged tile
__host__ __device__ constexpr int stage_stride(int cin) { return cin + (cin / 8 % 2 ? 0 : 8); }
// bytes of LDS: the tile, then eight zeros for the k beyond 9 cin
__host__ __device__ constexpr int stage_bytes(int th, int cin)
{
    return ((th + 2) * kHaloW * stage_stride(cin) + 8) * 2;
}

// q / d for 0 <= q < 2^16, 2 <= d < 2^16, r = ceil(2^32 / d) (d = 1: r = 0)
__device__ __forceinline__ int div_small(int q, unsigned r)
{
    return r ? (int)__umulhi((unsigned)q, r) : q;
}
__host__ __device__ constexpr unsigned div_recip(int d)
{
    return d > 1 ? (unsigned)(((1ull << 32) + d - 1) / d) : 0u;
}

// One image of an input, at the output resolution h x w.
struct Image {
    const __bf16 *x;
    int c, h, w;
};
__device__ __forceinline__ Image image_of(const In &in, int n, int h, int w)
{
    const long px = in.mode == kModePool ? 4l * h * w
                    : in.mode == kModeUp ? (long)(h >> 1) * (w >> 1)
                                         : (long)h * w;
    return Image{in.x + px * in.c * n, in.c, h, w};
}
// load_in's eight channels ci.. at pixel (y, x), zeros outside the image or
// without ok.  No branch: the image's first channels are read instead and
// dropped, so a lane's loads are all under way together.
template <int MODE>
__device__ __forceinline__ bf16x8 load_at(const Image &I, int ci, int y, int x, bool ok)
{
    typedef __attribute__((__vector_size__(16))) unsigned u32x4;
    ok = ok && (unsigned)y < (unsigned)I.h && (unsigned)x < (unsigned)I.w;
    bf16x8 v;
    if constexpr (MODE == kModePool) {
        const int wf = 2 * I.w;
        const __bf16 *p = I.x + (ok ? (2l * y * wf + 2 * x) * I.c + ci : 0l);
        const bf16x8 a = ld8(p), b = ld8(p + I.c), c = ld8(p + (long)wf * I.c),
                     d = ld8(p + (long)wf * I.c + I.c);
#pragma unroll
        for (int i = 0; i < 8; ++i)
            v[i] = (__bf16)((((float)a[i] + (float)b[i]) + ((float)c[i] + (float)d[i])) * 0.25f);
    } else if constexpr (MODE == kModeUp) {
        v = ld8(I.x + (ok ? ((long)(y >> 1) * (I.w >> 1) + (x >> 1)) * I.c + ci : 0l));
    } else {
        v = ld8(I.x + (ok ? ((long)y * I.w + x) * I.c + ci : 0l));
    }
    const unsigned keep = ok ? 0xffffffffu : 0u;
    return (bf16x8)((u32x4)v & keep);
}

// stage the groups of eight channels of one input, rows y0 - 1 .. y0 + TH,
// columns x0 - 1 .. x0 + 16, into tile (first pixel's first channel there),
// U groups of a lane under way together
template <int TH, int MODE>
__device__ __forceinline__ void stage_input(const Image &I, __bf16 *tile, unsigned rc8, int y0,
                                            int x0, int cs)
{
    constexpr int U = MODE == kModePool ? 2 : 4;
    const int c8 = I.c >> 3, total = (TH + 2) * kHaloW * c8;
    constexpr unsigned rw = div_recip(kHaloW);
    for (int q0 = threadIdx.x; q0 < total; q0 += 256 * U) {
        bf16x8 v[U];
        int at[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int q = q0 + 256 * u;
            const int px = div_small(q, rc8), cg = q - px * c8;
            const int ty = div_small(px, rw), tx = px - ty * kHaloW;
            at[u] = px * cs + 8 * cg;
            v[u] = load_at<MODE>(I, 8 * cg, y0 + ty - 1, x0 + tx - 1, q < total);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (q0 + 256 * u < total) *reinterpret_cast<bf16x8 *>(tile + at[u]) = v[u];
    }
}

template <int TH>
__device__ __forceinline__ void stage_tile(const ConvArgs &A, __bf16 *tile, int n, int y0, int x0,
                                           int cs)
{
    const Image I = image_of(A.in1, n, A.h, A.w_);
    if (A.in1.mode == kModePool)
        stage_input<TH, kModePool>(I, tile, A.rc1, y0, x0, cs);
    else if (A.in1.mode == kModeUp)
        stage_input<TH, kModeUp>(I, tile, A.rc1, y0, x0, cs);
    else
        stage_input<TH, kMode0>(I, tile, A.rc1, y0, x0, cs);
    if (A.in2.c)
        stage_input<TH, kMode0>(image_of(A.in2, n, A.h, A.w_), tile + A.in1.c, A.rc2, y0, x0, cs);
}

// C8 > 0: input channels / 8 known when compiled, so the taps' places in the
// tile are constants (with C8 a multiple of four the same for the whole
// wave, else one of four by the lane's group); 0: from A, computed for every
// 32 k.
template <int NT, int MT, int WP, int WC, int C8>
__global__ __launch_bounds__(256) void k_conv3x3_tile(ConvArgs A)
{
    static_assert(WP * WC == 4, "four waves");
    constexpr int TH = MT * WP;
    extern __shared__ __attribute__((aligned(16))) __bf16 tile[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wp = wave % WP, wc = wave / WP;
    const int row = blockIdx.x / A.tiles_x, x0 = (blockIdx.x - row * A.tiles_x) * kTileW;
    const int n = row / A.tiles_y, y0 = (row - n * A.tiles_y) * TH;
    const int c8 = C8 ? C8 : (A.in1.c + A.in2.c) >> 3, cs = stage_stride(8 * c8);
    const int zero_at = (TH + 2) * kHaloW * cs;
    const int co0 = (blockIdx.y * WC + wc) * 16 * NT;
    if (threadIdx.x == 0) *reinterpret_cast<bf16x8 *>(tile + zero_at) = zero8();
    stage_tile<TH>(A, tile, n, y0, x0, cs);

    const int px = lane & 15, kg = lane >> 4;
    f32x4 acc[NT][MT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    const __bf16 *wrow = A.w + (long)(co0 + px) * A.kpad + 8 * kg;
    const __bf16 *base = tile + (wp * MT * kHaloW + px) * cs;
    // place of the eight channels k = 8 k8 .. in the tile, from base
    auto place = [&](int k8) {
        const int tap = C8 ? k8 / (C8 ? C8 : 1) : div_small(k8, A.rc8);
        const int ky = C8 ? tap / 3 : (tap * 11) >> 5;  // tap / 3 for tap < 16
        return ((ky * kHaloW + (tap - 3 * ky)) * cs) + 8 * (k8 - tap * c8);
    };
    // weights are read AHEAD steps of 32 k before their products
    constexpr int AHEAD = 4;
    bf16x8 w[AHEAD][NT];
    auto fetch = [&](int slot, int kb) {
#pragma unroll
        for (int t = 0; t < NT; ++t) w[slot][t] = ld8(wrow + (long)t * 16 * A.kpad + kb);
    };
    auto step = [&](int slot, int off, bool some) {
        bf16x8 x[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) x[m] = ld8(some ? base + m * kHaloW * cs + off : tile + zero_at);
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int m = 0; m < MT; ++m)
                acc[t][m] =
                    __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[slot][t], x[m], acc[t][m], 0, 0, 0);
    };
    if constexpr (C8 == 0) {
        const int last = A.kpad - 32;
#pragma unroll
        for (int s = 0; s < AHEAD; ++s) fetch(s, 32 * s < last ? 32 * s : last);
        __syncthreads();
        for (int kb = 0; kb < A.kpad; kb += 32 * AHEAD) {
#pragma unroll
            for (int s = 0; s < AHEAD; ++s) {
                const int k = kb + 32 * s, k8 = (k >> 3) + kg;
                if (k < A.kpad) step(s, place(k8), k8 < 9 * c8);
                fetch(s, k + 32 * AHEAD < last ? k + 32 * AHEAD : last);
            }
        }
    } else {
        constexpr int STEPS = (72 * C8 + 31) / 32;
#pragma unroll
        for (int s = 0; s < AHEAD && s < STEPS; ++s) fetch(s, 32 * s);
        __syncthreads();
        if constexpr (C8 % 4 == 0) base += 8 * kg;
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            const int k8 = 4 * s;
            if constexpr (C8 % 4 == 0) {
                step(s % AHEAD, place(k8), true);
            } else {
                const int off = kg < 2 ? (kg == 0 ? place(k8) : place(k8 + 1))
                                       : (kg == 2 ? place(k8 + 2) : place(k8 + 3));
                step(s % AHEAD, off, k8 + 4 <= 9 * C8 || k8 + kg < 9 * C8);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (s + AHEAD < STEPS) fetch(s % AHEAD, 32 * (s + AHEAD));
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    const int xo = x0 + px;
    if (xo >= A.w_) return;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int co = co0 + 16 * t + 4 * kg;  // this lane's four channels
        if (co >= A.cout) continue;
        float bias[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) bias[i] = A.bias && co + i < A.cout ? A.bias[co + i] : 0.0f;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int yo = y0 + wp * MT + m;
            if (yo >= A.h) continue;
            const long o = (((long)n * A.h + yo) * A.w_ + xo) * A.cout_stride + co;
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[i] = acc[t][m][i] + bias[i];
                if (A.relu) v[i] = fmaxf(v[i], 0.0f);
            }
            if (A.vec) {  // four channels, aligned
                if (A.out) {
                    bf16x4 r;
#pragma unroll
                    for (int i = 0; i < 4; ++i) r[i] = (__bf16)v[i];
                    *reinterpret_cast<bf16x4 *>(A.out + o) = r;
                }
                if (A.out32) {
                    f32x4 *d = reinterpret_cast<f32x4 *>(A.out32 + o);
                    f32x4 r = {v[0], v[1], v[2], v[3]};
                    if (A.accumulate) r = *d + r;
                    *d = r;
                }
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (co + i >= A.cout) continue;
                    if (A.out) A.out[o + i] = (__bf16)v[i];
                    if (A.out32) A.out32[o + i] = A.accumulate ? A.out32[o + i] + v[i] : v[i];
                }
            }
        }
    }
}

// Weight gradient dW[co][k] += sum_p G[p][co] * im2col(p, k): M = output
// channels, N = k, K = pixels, so both operands want eight neighbouring
// pixels of one channel where the tensors hold eight channels of one pixel.
// A workgroup owns 16 input channels (all nine taps of them) and 16 MF output
// channels and goes through its share of the tiles of 16 x 16 pixels: it
// stages input and gradient transposed into LDS, and each wave adds two of the
// tile's rows (32 pixels) into 9 MF accumulators.  The three taps of a row
// come from one read of ten pixels, shifted in registers.  The next tile's
// loads are under way while a tile is computed.  At the end the waves'
// sums meet in LDS and leave with one FP32 atomic each.
//   bound: latency; a tile's transposing two-byte LDS writes, its reads and
// its products follow one another between barriers, and no unit is near its
// rate (258x130, 16 images: matrix cores busy for 4 to 7 % of a kernel's time,
// LDS for 10 to 16 %).  Before, every lane fetched every element of both
// operands from memory by itself.
constexpr int kGradH = 16, kGradWaves = kGradH / 2, kGradThreads = 64 * kGradWaves;
constexpr int kGradRow = 16 + 8;                      // pixels between two staged rows
constexpr int kGradX = (kGradH + 2) * kGradRow + 8;   // ... two channels (input)
constexpr int kGradG = kGradH * kTileW + 8;           // ... two channels (gradient)

// pixels p + 1 .. p + 8 of eight pixels p .. and the two after them
__device__ __forceinline__ bf16x8 shift_one(bf16x8 v, unsigned next)
{
    typedef __attribute__((__vector_size__(16))) unsigned u32x4;
    const u32x4 a = (u32x4)v;
    u32x4 r;
    r[0] = __builtin_amdgcn_alignbit(a[1], a[0], 16);
    r[1] = __builtin_amdgcn_alignbit(a[2], a[1], 16);
    r[2] = __builtin_amdgcn_alignbit(a[3], a[2], 16);
    r[3] = __builtin_amdgcn_alignbit(next, a[3], 16);
    return (bf16x8)r;
}
// pixels p + 2 .. p + 9
__device__ __forceinline__ bf16x8 shift_two(bf16x8 v, unsigned next)
{
    typedef __attribute__((__vector_size__(16))) unsigned u32x4;
    const u32x4 a = (u32x4)v;
    const u32x4 r = {a[1], a[2], a[3], next};
    return (bf16x8)r;
}

struct WgradArgs {
    ConvArgs c;          // inputs and geometry of the forward convolution
    const __bf16 *g;     // gradient at the convolution's output (pre-activation), cout channels
    float *dw;           // [cout_pad][kpad]
    float *db;           // cout values, or null
    int tiles_x, tiles_y, tiles;
};

// MODE: the first input's; VEC: cout a multiple of eight, g aligned
template <int MF, int MODE, bool VEC>
__global__ __launch_bounds__(kGradThreads, 4) void k_conv3x3_wgrad(WgradArgs W)
{
    constexpr int kStage = 16 * kGradX + 16 * MF * kGradG, kSums = 9 * MF * 64 * 8;
    constexpr int kLds = kStage > kSums ? kStage : kSums;
    __shared__ __attribute__((aligned(16))) __bf16 lds[kLds];
    __bf16 *const xt = lds, *const gt = lds + 16 * kGradX;
    const ConvArgs &A = W.c;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int ci0 = blockIdx.x * 16, co0 = blockIdx.y * 16 * MF;
    const int cin = A.in1.c + A.in2.c;
    const int l16 = lane & 15, kg = lane >> 4;
    f32x4 acc[9][MF];
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int m = 0; m < MF; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    float bsum[MF];
#pragma unroll
    for (int m = 0; m < MF; ++m) bsum[m] = 0.0f;
    const bool bias = W.db && blockIdx.x == 0;

    // what this thread stages of every tile: up to NX groups of eight input
    // channels of a halo pixel and NG of eight gradient channels of a pixel
    constexpr int kHalo = (kGradH + 2) * kHaloW;
    constexpr int NX = (2 * kHalo + kGradThreads - 1) / kGradThreads, NG = 2 * MF * kGradH * kTileW / kGradThreads;
    bf16x8 vx[NX], vg[NG];
    // the input that holds this workgroup's two groups: each thread's group
    // may lie in the first or in the second input
    auto fetch_x = [&](auto mode, int k, int n, int y0, int x0) {
        const int q = threadIdx.x + kGradThreads * k;
        const int cg = q / kHalo, px = q - cg * kHalo;
        const int sy = px / kHaloW, sx = px - sy * kHaloW;
        const int ci = ci0 + 8 * cg;
        const bool ok = q < 2 * kHalo && ci < cin;
        const int y = y0 + sy - 1, x = x0 + sx - 1;
        if (ci0 + 8 < A.in1.c || !A.in2.c) {
            vx[k] = load_at<decltype(mode)::value>(image_of(A.in1, n, A.h, A.w_), ci, y, x,
                                                   ok && ci < A.in1.c);
        } else if (ci0 >= A.in1.c) {
            vx[k] = load_at<kMode0>(image_of(A.in2, n, A.h, A.w_), ci - A.in1.c, y, x, ok);
        } else {  // one group of each
            const bf16x8 a = load_at<decltype(mode)::value>(image_of(A.in1, n, A.h, A.w_), ci, y, x,
                                                            ok && cg == 0);
            const bf16x8 b = load_at<kMode0>(image_of(A.in2, n, A.h, A.w_), 0, y, x, ok && cg == 1);
            vx[k] = cg == 0 ? a : b;
        }
    };
    auto fetch = [&](int tile) {
        const int n = tile / (W.tiles_x * W.tiles_y), r = tile - n * W.tiles_x * W.tiles_y;
        const int ty = r / W.tiles_x, y0 = ty * kGradH, x0 = (r - ty * W.tiles_x) * kTileW;
#pragma unroll
        for (int k = 0; k < NX; ++k) fetch_x(std::integral_constant<int, MODE>{}, k, n, y0, x0);
        const Image G = image_of(In{W.g, A.cout, kMode0}, n, A.h, A.w_);
#pragma unroll
        for (int k = 0; k < NG; ++k) {
            const int q = threadIdx.x + kGradThreads * k;
            const int cg = q / (kGradH * kTileW), px = q - cg * kGradH * kTileW;
            const int y = y0 + px / kTileW, x = x0 + px % kTileW, co = co0 + 8 * cg;
            if constexpr (VEC) {
                vg[k] = load_at<kMode0>(G, co, y, x, co < A.cout);
            } else {
                vg[k] = zero8();
                if (y < A.h && x < A.w_) {
                    const __bf16 *g = W.g + (((long)n * A.h + y) * A.w_ + x) * A.cout + co;
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        if (co + i < A.cout) vg[k][i] = g[i];
                }
            }
        }
    };
    fetch(blockIdx.z);  // gridDim.z <= tiles
    for (int tile = blockIdx.z; tile < W.tiles; tile += gridDim.z) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NX; ++k) {
            const int q = threadIdx.x + kGradThreads * k;
            const int cg = q / kHalo, px = q - cg * kHalo;
            const int sy = px / kHaloW, sx = px - sy * kHaloW;
            if (q < 2 * kHalo) {
                __bf16 *d = xt + 8 * cg * kGradX + sy * kGradRow + sx;
#pragma unroll
                for (int i = 0; i < 8; ++i) d[i * kGradX] = vx[k][i];
            }
        }
#pragma unroll
        for (int k = 0; k < NG; ++k) {
            const int q = threadIdx.x + kGradThreads * k;
            const int cg = q / (kGradH * kTileW), px = q - cg * kGradH * kTileW;
            __bf16 *d = gt + 8 * cg * kGradG + px;
#pragma unroll
            for (int i = 0; i < 8; ++i) d[i * kGradG] = vg[k][i];
        }
        __syncthreads();
        if (tile + gridDim.z < W.tiles) fetch(tile + gridDim.z);
        // this wave's rows 2 wave and 2 wave + 1; the lane's eight pixels
        const int row = 2 * wave + (kg >> 1), col = 8 * (kg & 1);
        bf16x8 g[MF];
#pragma unroll
        for (int m = 0; m < MF; ++m) {
            g[m] = ld8(gt + (16 * m + l16) * kGradG + row * kTileW + col);
            if (bias) {
#pragma unroll
                for (int i = 0; i < 8; ++i) bsum[m] += (float)g[m][i];
            }
        }
#pragma unroll
        for (int ky = 0; ky < 3; ++ky) {
            const __bf16 *p = xt + l16 * kGradX + (row + ky) * kGradRow + col;
            const bf16x8 x0 = ld8(p);
            const unsigned next = *reinterpret_cast<const unsigned *>(p + 8);
            const bf16x8 x1 = shift_one(x0, next), x2 = shift_two(x0, next);
#pragma unroll
            for (int m = 0; m < MF; ++m) {
                acc[3 * ky][m] =
                    __builtin_amdgcn_mfma_f32_16x16x32_bf16(g[m], x0, acc[3 * ky][m], 0, 0, 0);
                acc[3 * ky + 1][m] =
                    __builtin_amdgcn_mfma_f32_16x16x32_bf16(g[m], x1, acc[3 * ky + 1][m], 0, 0, 0);
                acc[3 * ky + 2][m] =
                    __builtin_amdgcn_mfma_f32_16x16x32_bf16(g[m], x2, acc[3 * ky + 2][m], 0, 0, 0);
            }
        }
    }
    // the other waves' sums into wave 0's
    f32x4 *const red = reinterpret_cast<f32x4 *>(lds);
    for (int src = 1; src < kGradWaves; ++src) {
        __syncthreads();
        if (wave == src) {
#pragma unroll
            for (int t = 0; t < 9; ++t)
#pragma unroll
                for (int m = 0; m < MF; ++m) red[(t * MF + m) * 64 + lane] = acc[t][m];
        }
        __syncthreads();
        if (wave == 0) {
#pragma unroll
            for (int t = 0; t < 9; ++t)
#pragma unroll
                for (int m = 0; m < MF; ++m) acc[t][m] += red[(t * MF + m) * 64 + lane];
        }
    }
    // D[m][n]: lane holds n = lane % 16 (ci), m = 4 (lane / 16) + i (co)
    if (wave == 0 && ci0 + l16 < cin) {
#pragma unroll
        for (int t = 0; t < 9; ++t)
#pragma unroll
            for (int m = 0; m < MF; ++m)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int co = co0 + 16 * m + 4 * kg + i;
                    if (co < A.cout)
                        atomicAdd(&W.dw[(long)co * A.kpad + t * cin + ci0 + l16], acc[t][m][i]);
                }
    }
    if (W.db && blockIdx.x == 0) {
        // lanes l, l+16, l+32, l+48 hold partial sums of channel co0 + l%16
        float *const rb = reinterpret_cast<float *>(lds);
        __syncthreads();
#pragma unroll
        for (int m = 0; m < MF; ++m) {
            float s = bsum[m];
            s += __shfl_xor(s, 16);
            s += __shfl_xor(s, 32);
            if (lane < 16) rb[wave * 16 * MF + 16 * m + lane] = s;
        }
        __syncthreads();
        if (threadIdx.x < 16 * MF && co0 + (int)threadIdx.x < A.cout) {
            float s = 0.0f;
            for (int k = 0; k < kGradWaves; ++k) s += rb[k * 16 * MF + threadIdx.x];
            atomicAdd(&W.db[co0 + threadIdx.x], s);
        }
    }
}

// Elementwise pieces of the backward pass.
// g <- g * (y > 0): gradient through the ReLU, from the activation y.
__global__ __launch_bounds__(256) void k_relu_bwd(__bf16 *g, const __bf16 *y, long n)
{
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i < n && !((float)y[i] > 0.0f)) g[i] = (__bf16)0.0f;
}

// Gradient of a fused input mode, from the gradient `gi` of the effective
// input (output resolution h x w, `cs` channels, first `c` of them belong to
// this input) into `dst` (the tensor's own resolution, c channels), added in
// FP32 into dst32.  Pool: each fine pixel gets a quarter; upsampling: a
// coarse pixel sums its four.
__global__ __launch_bounds__(256) void k_mode_bwd(const float *gi, int cs, int c0, int c,
                                                  int mode, int n, int h, int w, float *dst32)
{
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (mode == kModePool) {
        const int hf = 2 * h, wf = 2 * w;
        const long tot = (long)n * hf * wf * c;
        if (i >= tot) return;
        const int ch = (int)(i % c);
        const long px = i / c;
        const int x = (int)(px % wf), y = (int)((px / wf) % hf), b = (int)(px / ((long)wf * hf));
        dst32[i] += 0.25f * gi[(((long)b * h + y / 2) * w + x / 2) * cs + c0 + ch];
    } else if (mode == kModeUp) {
        const int hc = h / 2, wc = w / 2;
        const long tot = (long)n * hc * wc * c;
        if (i >= tot) return;
        const int ch = (int)(i % c);
        const long px = i / c;
        const int x = (int)(px % wc), y = (int)((px / wc) % hc), b = (int)(px / ((long)wc * hc));
        float s = 0.0f;
        for (int dy = 0; dy < 2; ++dy)
            for (int dx = 0; dx < 2; ++dx)
                s += gi[(((long)b * h + 2 * y + dy) * w + 2 * x + dx) * cs + c0 + ch];
        dst32[i] += s;
    } else {
        const long tot = (long)n * h * w * c;
        if (i >= tot) return;
        const int ch = (int)(i % c);
        dst32[i] += gi[(i / c) * cs + c0 + ch];
    }
}

// bf16 copy of an FP32 tensor.
__global__ __launch_bounds__(256) void k_to_bf16(const float *src, __bf16 *dst, long n)
{
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = (__bf16)src[i];
}

// Gradient of a layer's pre-activation output (bf16) from the FP32 gradients
// of the one or two convolution inputs its activation y went into, each
// carried back through its mode to y's resolution h x w as k_mode_bwd does,
// added in their order, rounded and cut where y is not positive.  One pass
// over memory where zeroing, adding, rounding and the ReLU were four; a
// thread takes eight channels.
struct GradSrc {
    const float *g;  // null: none
    int cs, c0, mode;
};
struct GradArgs {
    GradSrc src[2];
    const __bf16 *y;
    __bf16 *out;
    int c, h, w;
    long groups;  // pixels * c / 8
};
__global__ __launch_bounds__(256) void k_grad_in(GradArgs A)
{
    const long q = (long)blockIdx.x * 256 + threadIdx.x;
    if (q >= A.groups) return;
    const int c8 = A.c >> 3;
    const long px = q / c8;
    const int ch = 8 * (int)(q - px * c8);
    const long row = px / A.w;
    const int x = (int)(px - row * A.w);
    const long n = row / A.h;
    const int y = (int)(row - n * A.h);
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = 0.0f;
    auto add = [&](const float *p, float f) {
        const f32x4 a = *reinterpret_cast<const f32x4 *>(p), b = *reinterpret_cast<const f32x4 *>(p + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] += f * a[i];
            v[4 + i] += f * b[i];
        }
    };
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const GradSrc &S = A.src[k];
        if (!S.g) continue;
        const float *g = S.g + S.c0 + ch;
        if (S.mode == kModePool) {
            add(g + ((n * (A.h >> 1) + (y >> 1)) * (A.w >> 1) + (x >> 1)) * S.cs, 0.25f);
        } else if (S.mode == kModeUp) {
            const float *p = g + ((n * 2 * A.h + 2 * y) * 2 * A.w + 2 * x) * S.cs;
            float t[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                t[i] = v[i];
                v[i] = 0.0f;
            }
            add(p, 1.0f);
            add(p + S.cs, 1.0f);
            add(p + 2l * A.w * S.cs, 1.0f);
            add(p + 2l * A.w * S.cs + S.cs, 1.0f);
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = t[i] + v[i];
        } else {
            add(g + px * S.cs, 1.0f);
        }
    }
    const bf16x8 act = ld8(A.y + px * A.c + ch);
    bf16x8 r;
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = (float)act[i] > 0.0f ? (__bf16)v[i] : (__bf16)0.0f;
    *reinterpret_cast<bf16x8 *>(A.out + px * A.c + ch) = r;
}

// Adam on FP32 master weights w[cout_pad][kpad] (and bias), then the bf16
// copies the kernels read: wb (same layout) and wr, the input-gradient
// weights [cin_pad][kpad_r] with wr[ci][tap' * cout + co] = w[co][(8 - tap') * cin + ci].
struct AdamArgs {
    float *w, *m, *v;
    const float *g;
    long n;
    float lr, b1, b2, eps, c1, c2;  // c1 = 1 - b1^t, c2 = 1 - b2^t
};

__global__ __launch_bounds__(256) void k_adam(AdamArgs a)
{
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= a.n) return;
    const float g = a.g[i];
    const float m = a.b1 * a.m[i] + (1.0f - a.b1) * g;
    const float v = a.b2 * a.v[i] + (1.0f - a.b2) * g * g;
    a.m[i] = m;
    a.v[i] = v;
    a.w[i] -= a.lr * (m / a.c1) / (sqrtf(v / a.c2) + a.eps);
}

// one layer per grid row
constexpr int kPackLayers = 24;
struct PackArgs {
    m2d_unet_layer l[kPackLayers];
};
__global__ __launch_bounds__(256) void k_pack_weights(PackArgs A)
{
    const m2d_unet_layer &P = A.l[blockIdx.y];
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    const long nw = (long)P.cout * P.kpad;
    __bf16 *const wb = (__bf16 *)P.wb, *const wr = (__bf16 *)P.wr;
    if (i < nw) wb[i] = (__bf16)P.w[i];
    if (wr && i < (long)P.cin_pad * P.kpad_r) {
        const int ci = (int)(i / P.kpad_r), k = (int)(i % P.kpad_r);
        float v = 0.0f;
        if (ci < P.cin && k < 9 * P.cout) {
            const int tr = k / P.cout, co = k - tr * P.cout;
            v = P.w[(long)co * P.kpad + (8 - tr) * P.cin + ci];
        }
        wr[i] = (__bf16)v;
    }
}

// Loss 0.5 * sum over masked pixels of (pred - target)^2 / count (1 / count
// from inv_count, or from the count in device memory, 0 for a count of 0), its
// gradient (bf16, `cs` channels with the value in channel 0) and per-block
// partial sums of the loss.
__global__ __launch_bounds__(256) void k_mse(const float *pred, int ps, const float *target,
                                             const float *mask, long npix, float inv_count,
                                             const float *count, __bf16 *grad, int gs,
                                             float *partial)
{
    if (count) inv_count = *count != 0.0f ? (float)(1.0 / (double)*count) : 0.0f;
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    float l = 0.0f;
    if (i < npix) {
        const float d = (pred[i * ps] - target[i]) * mask[i];
        l = 0.5f * d * d * inv_count;
        grad[i * gs] = (__bf16)(d * inv_count);
        for (int c = 1; c < gs; ++c) grad[i * gs + c] = (__bf16)0.0f;
    }
    __shared__ float red[256];
    red[threadIdx.x] = l;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// Network input from a 9-diagonal system (FP64, reference layout) and its
// right-hand side: the Jacobi-scaled form  p - sum (a_nb/a_P) p_nb = b/a_P.
// Channels: 0 b/(a_P s), 1..4 a_W, a_E, a_S, a_N over a_P, 5 the corner sum
// over a_P, 6..7 zero; s = RMS of b/a_P over the grid.  Pixels beyond the
// grid (the tensor is h x w >= ny x nx) are zero, as are fictitious rows
// with a_P = 0.
__global__ __launch_bounds__(256) void k_pack_input(const double *a, const double *b, int nx,
                                                    int ny, int h, int w, double inv_s,
                                                    __bf16 *x, int nb)
{
    const long q = (long)blockIdx.x * 256 + threadIdx.x;
    const long np_ = (long)h * w;
    if (q >= np_ * nb) return;
    const int bi = (int)(q / np_);
    const long pix = q - (long)bi * np_;
    const int xx = (int)(pix % w), yy = (int)(pix / w);
    float f[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (xx < nx && yy < ny) {
        const long N = (long)nx * ny, p = (long)yy * nx + xx;
        const double *as = a + (long)bi * 9 * N, *bs = b + (long)bi * N;
        const double ap = as[kP * N + p];
        if (ap != 0.0) {
            const double r = 1.0 / ap;
            f[0] = (float)(bs[p] * r * inv_s);
            f[1] = (float)(as[kW * N + p] * r);
            f[2] = (float)(as[kE * N + p] * r);
            f[3] = (float)(as[kS * N + p] * r);
            f[4] = (float)(as[kN * N + p] * r);
            f[5] = (float)((as[kSW * N + p] + as[kSE * N + p] + as[kNW * N + p] +
                            as[kNE * N + p]) * r);
        }
    }
    bf16x8 v;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = (__bf16)f[i];
    *reinterpret_cast<bf16x8 *>(x + q * 8) = v;
}

// Guess var = s * out (channel 0 of the FP32 output) on the grid.
__global__ __launch_bounds__(256) void k_unpack_output(const float *out, int os, int nx, int ny,
                                                       int w, double s, double *var)
{
    const long q = (long)blockIdx.x * 256 + threadIdx.x;
    if (q >= (long)nx * ny) return;
    const int xx = (int)(q % nx), yy = (int)(q / nx);
    var[q] = s * (double)out[((long)yy * w + xx) * os];
}

}  // namespace unet
}  // namespace m2d

using namespace m2d;
using namespace m2d::unet;

namespace {
unsigned blocks256(long n) { return (unsigned)((n + 255) / 256); }
int rc_of(hipError_t e) { return e == hipSuccess ? M2D_OK : M2D_ERR_HIP; }
bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

template <int MF, int MODE>
void launch_wgrad_mode(const WgradArgs &W, bool vec, dim3 grid, hipStream_t s)
{
    if (vec)
        hipLaunchKernelGGL((k_conv3x3_wgrad<MF, MODE, true>), grid, dim3(kGradThreads), 0, s, W);
    else
        hipLaunchKernelGGL((k_conv3x3_wgrad<MF, MODE, false>), grid, dim3(kGradThreads), 0, s, W);
}
template <int MF>
void launch_wgrad(const WgradArgs &W, bool vec, dim3 grid, hipStream_t s)
{
    if (W.c.in1.mode == kModePool)
        launch_wgrad_mode<MF, kModePool>(W, vec, grid, s);
    else if (W.c.in1.mode == kModeUp)
        launch_wgrad_mode<MF, kModeUp>(W, vec, grid, s);
    else
        launch_wgrad_mode<MF, kMode0>(W, vec, grid, s);
}

// Rows of a tile with 16, 32, 64 output channels per workgroup (nt = 1, 2,
// 4): mt for each of the waves along the rows
constexpr int tile_rows(int nt, int mt) { return nt == 4 ? 2 * mt : 4 * mt; }

template <int NT, int MT, int WP, int WC, int C8, int... More>
void launch_conv_c8(const ConvArgs &A, dim3 grid, int lds, hipStream_t s)
{
    if constexpr (sizeof...(More) > 0)
        if (A.in1.c + A.in2.c != 8 * C8)
            return launch_conv_c8<NT, MT, WP, WC, More...>(A, grid, lds, s);
    hipLaunchKernelGGL((k_conv3x3_tile<NT, MT, WP, WC, C8>), grid, dim3(256), lds, s, A);
}

// the channel counts of the network's layers and their input gradients, any
// other with computed places
template <int MT>
void launch_conv_tile(const ConvArgs &A, int nt, dim3 grid, int lds, hipStream_t s)
{
    if (nt == 4)
        launch_conv_c8<2, MT, 2, 2, 4, 8, 16, 24, 0>(A, grid, lds, s);
    else if (nt == 2)
        launch_conv_c8<2, MT, 4, 1, 2, 4, 8, 12, 0>(A, grid, lds, s);
    else
        launch_conv_c8<1, MT, 4, 1, 1, 2, 4, 6, 0>(A, grid, lds, s);
}
}  // namespace

// ---------------------------------------------------------------------------
// C ABI (device pointers, stream as void*).  No reference counterpart.
// ---------------------------------------------------------------------------

extern "C" int m2d_unet_conv3x3(const void *in1, int c1, int mode1, const void *in2, int c2,
                                const void *w, const float *bias, int cout, int cout_stride,
                                int kpad, int n, int h, int w_, int relu, void *out,
                                float *out32, int accumulate, void *stream)
{
    const int cin = c1 + c2;
    if (!in1 || c1 <= 0 || c1 % 8 || c2 < 0 || c2 % 8 || (c2 && !in2) || !w || cout <= 0 ||
        cout_stride < cout || kpad < 9 * cin || kpad % 32 || n <= 0 || h <= 0 || w_ <= 0 ||
        (!out && !out32) || mode1 < 0 || mode1 > 2 || (mode1 == kModeUp && (h % 2 || w_ % 2)))
        return M2D_ERR_ARG;
    if (!aligned16(in1) || (in2 && !aligned16(in2)) || !aligned16(w)) return M2D_ERR_ARG;
    ConvArgs A;
    A.in1 = In{(const __bf16 *)in1, c1, mode1};
    A.in2 = In{(const __bf16 *)in2, c2, kMode0};
    A.w = (const __bf16 *)w;
    A.bias = bias;
    A.out = (__bf16 *)out;
    A.out32 = out32;
    A.cout = cout;
    A.cout_stride = cout_stride;
    A.kpad = kpad;
    A.n = n;
    A.h = h;
    A.w_ = w_;
    A.relu = relu;
    A.accumulate = accumulate;
    const long npix = (long)n * h * w_;
    if (npix > 0x7fffffffL / 2) return M2D_ERR_ARG;
    A.vec = cout % 4 == 0 && cout_stride % 4 == 0 && ((uintptr_t)out & 7) == 0 &&
            ((uintptr_t)out32 & 15) == 0;
    const int cpad = (cout + 15) / 16 * 16;  // weight rows available: cout rounded to 16
    const hipStream_t s = (hipStream_t)stream;
    // 64 channels per workgroup where the weights have them (the input is
    // staged once for all of them), else 32, else 16
    const int nt = cpad % 64 == 0 ? 4 : cpad % 32 == 0 ? 2 : 1;
    // Four rows of the tile per wave where its LDS allows and that leaves two
    // workgroups for every CU (one with 64 channels, whose weights' reads
    // from L2 are what the taller tile halves), else two
    const long fill = nt == 4 ? 256 : 512;
    A.tiles_x = (w_ + kTileW - 1) / kTileW;
    for (int mt = 4; mt >= 2; mt -= 2) {
        const int th = tile_rows(nt, mt), lds = stage_bytes(th, cin);
        A.tiles_y = (h + th - 1) / th;
        const long tiles = (long)A.tiles_x * A.tiles_y * n;  // below npix
        const dim3 g((unsigned)tiles, (unsigned)(cpad / (16 * nt)));
        if (lds > (mt == 4 ? 80 : 64) * 1024 || (mt == 4 && (long)g.x * g.y < fill)) continue;
        A.rc8 = div_recip(cin / 8);
        A.rc1 = div_recip(c1 / 8);
        A.rc2 = c2 ? div_recip(c2 / 8) : 0;
        if (mt == 4)
            launch_conv_tile<4>(A, nt, g, lds, s);
        else
            launch_conv_tile<2>(A, nt, g, lds, s);
        return rc_of(hipGetLastError());
    }
    dim3 grid((unsigned)((npix + 63) / 64), (unsigned)(cpad / (16 * nt)));
    if (nt == 4)
        hipLaunchKernelGGL(k_conv3x3<4>, grid, dim3(256), 0, s, A);
    else if (nt == 2)
        hipLaunchKernelGGL(k_conv3x3<2>, grid, dim3(256), 0, s, A);
    else
        hipLaunchKernelGGL(k_conv3x3<1>, grid, dim3(256), 0, s, A);
    return rc_of(hipGetLastError());
}

extern "C" int m2d_unet_conv3x3_wgrad(const void *in1, int c1, int mode1, const void *in2, int c2,
                                      const void *g, int cout, int kpad, int n, int h, int w_,
                                      float *dw, float *db, void *stream)
{
    const int cin = c1 + c2;
    if (!in1 || c1 <= 0 || c1 % 8 || c2 < 0 || c2 % 8 || (c2 && !in2) || !g || !dw ||
        cout <= 0 || kpad < 9 * cin || kpad % 32 || n <= 0 || h <= 0 || w_ <= 0 ||
        mode1 < 0 || mode1 > 2 || (mode1 == kModeUp && (h % 2 || w_ % 2)))
        return M2D_ERR_ARG;
    WgradArgs W;
    W.c.in1 = In{(const __bf16 *)in1, c1, mode1};
    W.c.in2 = In{(const __bf16 *)in2, c2, kMode0};
    W.c.cout = cout;
    W.c.kpad = kpad;
    W.c.n = n;
    W.c.h = h;
    W.c.w_ = w_;
    W.g = (const __bf16 *)g;
    W.dw = dw;
    W.db = db;
    W.tiles_x = (w_ + kTileW - 1) / kTileW;
    W.tiles_y = (h + kGradH - 1) / kGradH;
    const long tiles = (long)W.tiles_x * W.tiles_y * n;
    if (tiles > 0x7fffffffL) return M2D_ERR_ARG;
    W.tiles = (int)tiles;
    // 32 output channels per workgroup where there are as many (64 took 312
    // registers a lane: one wave per SIMD), and two workgroups of eight waves
    // for every CU, but at most 256 on the same outputs: their atomics meet
    // there (16 x 16 channels: 29 us with 256, 61 with 1024, 113 with 2048)
    // and each adds a rounding
    const int mf = cout > 16 ? 2 : 1;
    const int gx = (cin + 15) / 16, gy = (cout + 16 * mf - 1) / (16 * mf);
    long gz = (512 + gx * gy - 1) / (gx * gy);
    gz = gz < 256 ? gz : 256;
    gz = gz < tiles ? gz : tiles;
    const dim3 grid((unsigned)gx, (unsigned)gy, (unsigned)gz);
    const hipStream_t s = (hipStream_t)stream;
    const bool vec = cout % 8 == 0 && aligned16(g);
    if (mf == 2)
        launch_wgrad<2>(W, vec, grid, s);
    else
        launch_wgrad<1>(W, vec, grid, s);
    return rc_of(hipGetLastError());
}

extern "C" int m2d_unet_relu_bwd(void *g, const void *y, long count, void *stream)
{
    if (!g || !y || count < 0) return M2D_ERR_ARG;
    if (!count) return M2D_OK;
    hipLaunchKernelGGL(k_relu_bwd, dim3(blocks256(count)), dim3(256), 0, (hipStream_t)stream,
                       (__bf16 *)g, (const __bf16 *)y, count);
    return rc_of(hipGetLastError());
}

extern "C" int m2d_unet_mode_bwd(const float *gi, int cs, int c0, int c, int mode, int n, int h,
                                 int w, float *dst32, void *stream)
{
    if (!gi || !dst32 || c <= 0 || c0 < 0 || c0 + c > cs || mode < 0 || mode > 2) return M2D_ERR_ARG;
    const long tot = mode == kModePool  ? (long)n * 4 * h * w * c
                     : mode == kModeUp ? (long)n * (h / 2) * (w / 2) * c
                                       : (long)n * h * w * c;
    hipLaunchKernelGGL(k_mode_bwd, dim3(blocks256(tot)), dim3(256), 0, (hipStream_t)stream, gi,
                       cs, c0, c, mode, n, h, w, dst32);
    return rc_of(hipGetLastError());
}

extern "C" int m2d_unet_to_bf16(const float *src, void *dst, long count, void *stream)
{
    if (!src || !dst || count < 0) return M2D_ERR_ARG;
    if (!count) return M2D_OK;
    hipLaunchKernelGGL(k_to_bf16, dim3(blocks256(count)), dim3(256), 0, (hipStream_t)stream, src,
                       (__bf16 *)dst, count);
    return rc_of(hipGetLastError());
}

extern "C" int m2d_unet_adam(float *w, float *m, float *v, const float *g, long count, float lr,
                             float b1, float b2, float eps, int step, void *stream)
{
    if (!w || !m || !v || !g || count < 0 || step < 1) return M2D_ERR_ARG;
    if (!count) return M2D_OK;
    AdamArgs a{w, m, v, g, count, lr, b1, b2, eps, 1.0f - powf(b1, (float)step),
               1.0f - powf(b2, (float)step)};
    hipLaunchKernelGGL(k_adam, dim3(blocks256(count)), dim3(256), 0, (hipStream_t)stream, a);
    return rc_of(hipGetLastError());
}

extern "C" int m2d_unet_pack_weights_many(int count, const m2d_unet_layer *layers, void *stream)
{
    if (count < 0 || (count && !layers)) return M2D_ERR_ARG;
    for (int k = 0; k < count; ++k) {
        const m2d_unet_layer &l = layers[k];
        if (!l.w || !l.wb || l.cout <= 0 || l.cin <= 0 || l.kpad < 9 * l.cin ||
            (l.wr && (l.kpad_r < 9 * l.cout || l.cin_pad < l.cin)))
            return M2D_ERR_ARG;
    }
    for (int k0 = 0; k0 < count; k0 += kPackLayers) {
        const int m = count - k0 < kPackLayers ? count - k0 : kPackLayers;
        PackArgs A;
        long most = 1;
        for (int k = 0; k < m; ++k) {
            const m2d_unet_layer &l = A.l[k] = layers[k0 + k];
            const long nw = (long)l.cout * l.kpad, nr = l.wr ? (long)l.cin_pad * l.kpad_r : 0;
            most = nw > most ? nw : most;
            most = nr > most ? nr : most;
        }
        hipLaunchKernelGGL(k_pack_weights, dim3(blocks256(most), (unsigned)m), dim3(256), 0,
                           (hipStream_t)stream, A);
    }
    return rc_of(hipGetLastError());
}

extern "C" int m2d_unet_pack_weights(const float *w, int cout, int cin, int kpad, void *wb,
                                     void *wr, int kpad_r, int cin_pad, void *stream)
{
    const m2d_unet_layer l = {w, wb, wr, cout, cin, kpad, kpad_r, cin_pad};
    return m2d_unet_pack_weights_many(1, &l, stream);
}

extern "C" int m2d_unet_grad_in(const float *g1, int cs1, int c01, int mode1, const float *g2,
                                int cs2, int c02, int mode2, const void *y, int c, int n, int h,
                                int w, void *out, void *stream)
{
    if (!g1 || !y || !out || c <= 0 || c % 8 || n <= 0 || h <= 0 || w <= 0) return M2D_ERR_ARG;
    GradArgs A;
    A.src[0] = GradSrc{g1, cs1, c01, mode1};
    A.src[1] = GradSrc{g2, cs2, c02, mode2};
    for (const GradSrc &S : A.src)
        if (S.g && (S.mode < 0 || S.mode > 2 || S.c0 < 0 || S.c0 % 4 || S.cs % 4 ||
                    S.c0 + c > S.cs || !aligned16(S.g) ||
                    (S.mode == kModePool && (h % 2 || w % 2))))
            return M2D_ERR_ARG;
    if (!aligned16(y) || !aligned16(out)) return M2D_ERR_ARG;
    A.y = (const __bf16 *)y;
    A.out = (__bf16 *)out;
    A.c = c;
    A.h = h;
    A.w = w;
    A.groups = (long)n * h * w * (c / 8);
    hipLaunchKernelGGL(k_grad_in, dim3(blocks256(A.groups)), dim3(256), 0, (hipStream_t)stream, A);
    return rc_of(hipGetLastError());
}

static int mse(const float *pred, int ps, const float *target, const float *mask, long npix,
               float inv_count, const float *count, void *grad, int gs, float *partial,
               void *stream)
{
    if (!pred || !target || !mask || !grad || !partial || npix <= 0 || ps < 1 || gs < 1)
        return M2D_ERR_ARG;
    hipLaunchKernelGGL(k_mse, dim3(blocks256(npix)), dim3(256), 0, (hipStream_t)stream, pred, ps,
                       target, mask, npix, inv_count, count, (__bf16 *)grad, gs, partial);
    return rc_of(hipGetLastError());
}

extern "C" int m2d_unet_mse(const float *pred, int ps, const float *target, const float *mask,
                            long npix, float inv_count, void *grad, int gs, float *partial,
                            void *stream)
{
    return mse(pred, ps, target, mask, npix, inv_count, nullptr, grad, gs, partial, stream);
}

extern "C" int m2d_unet_mse_count(const float *pred, int ps, const float *target,
                                  const float *mask, long npix, const float *count, void *grad,
                                  int gs, float *partial, void *stream)
{
    if (!count) return M2D_ERR_ARG;
    return mse(pred, ps, target, mask, npix, 0.0f, count, grad, gs, partial, stream);
}

extern "C" int m2d_unet_pack_input(const double *a, const double *b, int nx, int ny, int h, int w,
                                   double inv_s, void *x, int nb, void *stream)
{
    if (!a || !b || !x || nx <= 0 || ny <= 0 || h < ny || w < nx || nb <= 0) return M2D_ERR_ARG;
    hipLaunchKernelGGL(k_pack_input, dim3(blocks256((long)h * w * nb)), dim3(256), 0,
                       (hipStream_t)stream, a, b, nx, ny, h, w, inv_s, (__bf16 *)x, nb);
    return rc_of(hipGetLastError());
}

extern "C" int m2d_unet_unpack_output(const float *out, int os, int nx, int ny, int w, double s,
                                      double *var, void *stream)
{
    if (!out || !var || nx <= 0 || ny <= 0 || w < nx || os < 1) return M2D_ERR_ARG;
    hipLaunchKernelGGL(k_unpack_output, dim3(blocks256((long)nx * ny)), dim3(256), 0,
                       (hipStream_t)stream, out, os, nx, ny, w, s, var);
    return rc_of(hipGetLastError());
}
