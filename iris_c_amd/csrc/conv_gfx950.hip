/*
 * Convolutions of a channels-last f32 image that need neither a patch matrix nor a bf16 copy of the image
 * (reference iris_dev.h:111-121, iris_cuda.cu:959-1016; the other shapes are in gemm_conv_gfx950.hip).
 *
 * k_conv_few_in: k * k * cin <= 32, the 3-channel input of the VAE encoder.
 * k_conv_few_out: k * k * cout <= 28, the 3-channel output of the VAE decoder.
 *
 * Both are bound by memory: one side of the product is so thin that the image on the other side is all there is to
 * move. The image is rounded to bf16 on the way into the matrix core, products are summed in f32.
 */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "iris_kernels_hip.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

namespace {

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    f32x2 p = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(p, bf16x2));
}
__device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

struct ConvShape {
    int h, w, cin, cout, k, stride, pad, oh, ow;      /* pad: rows and columns of zeros in front; ow, oh: output size */
};

/* ---- few input channels ----
 *
 * The whole patch of an output pixel, k * k * cin <= 32 values, is one k-step of v_mfma_f32_16x16x32_bf16: A = 16
 * output channels, B = 16 pixels. A wave keeps the weights of 128 output channels (eight A operands) in
 * registers and walks groups of 16 consecutive pixels: a lane gathers its eight patch values (cached: neighbouring
 * pixels share them), eight products, and the 16 x 128 results leave through the LDS as whole 512-byte rows.
 * What bounds it is the output stream. 3 -> 128 on 512 x 512 (134 MB out): 902 us as patches + scalar product + bias,
 * 40 us here (3.4 TB/s). */
constexpr int FI_WAVES = 4, FI_COLS = 128;

template <bool ALIGNED>
__global__ void __launch_bounds__(64 * FI_WAVES, 4)
k_conv_few_in(float *__restrict__ out, const float *__restrict__ in, const uint16_t *__restrict__ W, const float *__restrict__ bias,
              ConvShape s, int groups) {
    __shared__ __align__(16) float lds[FI_WAVES * 16 * FI_COLS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, lg = lane >> 4;
    const int n0 = blockIdx.y * FI_COLS, row_len = s.k * s.k * s.cin, pixels = s.oh * s.ow;
    float *buf = lds + wave * 16 * FI_COLS;

    u32x4 av[8];
#pragma unroll
    for (int a = 0; a < 8; a++) {
        const int n = n0 + 16 * a + li;
        uint16_t e[8];
#pragma unroll
        for (int j = 0; j < 8; j++) e[j] = n < s.cout && 8 * lg + j < row_len ? W[(size_t)n * row_len + 8 * lg + j] : (uint16_t)0;
        av[a] = u32x4{e[0] | (uint32_t)e[1] << 16, e[2] | (uint32_t)e[3] << 16, e[4] | (uint32_t)e[5] << 16, e[6] | (uint32_t)e[7] << 16};
    }
    f32x4 bv = {0, 0, 0, 0};                                   /* of the four channels this lane stores */
    for (int r = 0; r < 4; r++)
        if (bias && n0 + 4 * (lane & 31) + r < s.cout) bv[r] = bias[n0 + 4 * (lane & 31) + r];
    /* patch value 8 lg + j of a pixel: (dy, dx) of its tap and its offset from the patch's first value */
    int dy[8], dx[8], off[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const int r = 8 * lg + j, tap = r / s.cin, c = r - tap * s.cin;
        dy[j] = r < row_len ? tap / s.k : 1 << 28;              /* beyond the patch: never inside the image */
        dx[j] = tap % s.k;
        off[j] = (tap / s.k * s.w + dx[j]) * s.cin + c;
    }

    float v[8];
    auto fetch = [&](int g) {
        const int p = 16 * g + li;
        const int oy = p / s.ow, y0 = oy * s.stride - s.pad, x0 = (p - oy * s.ow) * s.stride - s.pad;
        const long base = ((long)y0 * s.w + x0) * s.cin;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int y = y0 + dy[j], x = x0 + dx[j];
            const bool inside = p < pixels && (unsigned)y < (unsigned)s.h && (unsigned)x < (unsigned)s.w;
            const float t = in[inside ? base + off[j] : 0];
            v[j] = inside ? t : 0.0f;
        }
    };
    int g = blockIdx.x * FI_WAVES + wave;
    if (g < groups) fetch(g);
    for (; g < groups; g += gridDim.x * FI_WAVES) {
        const u32x4 b = {pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7])};
        /* lane: channels 16 a + 4 lg .. + 3 of pixel li. 16-byte chunk c of pixel r in slot (c & 16) | ((c ^ r) & 15): the
         * writes (16 pixels, one chunk) and the reads (32 chunks of a pixel) both spread over all banks. A wave's own
         * region, and the LDS serves a wave's instructions in order: no barrier. */
#pragma unroll
        for (int a = 0; a < 8; a++) {
            const int chunk = 4 * a + lg;
            *reinterpret_cast<f32x4 *>(&buf[li * FI_COLS + 4 * ((chunk & 16) | ((chunk ^ li) & 15))]) = mfma(av[a], b, f32x4{0, 0, 0, 0});
        }
        if (g + gridDim.x * FI_WAVES < groups) fetch(g + gridDim.x * FI_WAVES);     /* on its way while this group is stored */
#pragma unroll
        for (int it = 0; it < 8; it++) {
            const int row = 2 * it + (lane >> 5), c = lane & 31, m = 16 * g + row, n = n0 + 4 * c;
            const f32x4 r = *reinterpret_cast<const f32x4 *>(&buf[row * FI_COLS + 4 * ((c & 16) | ((c ^ row) & 15))]) + bv;
            float *dst = out + (size_t)m * s.cout + n;
            if (m >= pixels) continue;
            if (ALIGNED) {
                if (n < s.cout) *reinterpret_cast<f32x4 *>(dst) = r;
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (n + e < s.cout) dst[e] = r[e];
            }
        }
    }
}

/* ---- few output channels ----
 *
 * The taps move from the reduction into the rows of the product: Z[(tap, channel)][pixel] = W[channel, tap] . image[pixel]
 * for every INPUT pixel, k * k * cout <= 28 rows (two A operands), cin long; the output pixel then adds its k * k entries of
 * Z. So a pixel goes through the matrix core once instead of once per tap, its B operand comes straight from global
 * memory (a k-step's 32 channels as two 16-byte loads a lane, channels 4 lg and 16 + 4 lg, so that a load covers 64 B of a pixel), and only Z passes through the LDS. A workgroup makes Z for the
 * (32 + k - 1) x (16 + k - 1) pixels under a 32 x 16 tile of the output (1.2 x, the overlap comes from the L2).
 * What bounds it is the read of the image. 128 -> 3 on 1024 x 1024 (537 MB in): 1383 us as patches + 128-wide product +
 * bias, 122 us here (5.3 TB/s with the overlap). Two workgroups per CU (Z and the weights take 78 KB of LDS), so that one adds while one reads. */
constexpr int FO_TX = 32, FO_TY = 16, FO_THREADS = 512, FO_ROWS = 28, FO_MAX_K = 3;
constexpr int FO_PIXELS = (FO_TX + FO_MAX_K - 1) * (FO_TY + FO_MAX_K - 1), FO_MAX_CIN = 128;
constexpr int FO_GROUPS = (FO_PIXELS + 15) / 16;
constexpr int FO_LDS = FO_GROUPS * 16 * FO_ROWS * 4 + 2 * (FO_MAX_CIN / 32) * 1024;

template <int STEPS>                                         /* cin / 32 */
__global__ void __launch_bounds__(FO_THREADS, 4)
k_conv_few_out(float *__restrict__ out, const float *__restrict__ in, const uint16_t *__restrict__ W, const float *__restrict__ bias,
               ConvShape s, int tiles_x, int tiles, int per_xcd) {
    extern __shared__ __align__(16) float z[];               /* [pixel of the tile with its rim][FO_ROWS], then the weights */
    u32x4 *wf = reinterpret_cast<u32x4 *>(z + FO_GROUPS * 16 * FO_ROWS);      /* A operands: [k-step][2][64 lanes] */
    /* tiles that share rows of the image run on the same XCD: each XCD takes a contiguous range of them */
    const int work = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (work >= tiles) return;
    const int ty0 = work / tiles_x * FO_TY, tx0 = work % tiles_x * FO_TX;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, lg = lane >> 4;
    const int taps = s.k * s.k, hx = FO_TX + s.k - 1, pixels = hx * (FO_TY + s.k - 1), groups = (pixels + 15) / 16;

    for (int i = threadIdx.x; i < STEPS * 128; i += FO_THREADS) {
        const int row = 16 * ((i >> 6) & 1) + (i & 15), ks = i >> 7, g = (i >> 4) & 3;
        const int tap = row / s.cout, co = row - tap * s.cout;
        u32x4 v = {0, 0, 0, 0};
        if (tap < taps) {
            const uint16_t *src = W + ((size_t)co * taps + tap) * s.cin + 32 * ks + 4 * g;
            const uint2 lo = *reinterpret_cast<const uint2 *>(src), hi = *reinterpret_cast<const uint2 *>(src + 16);
            v = u32x4{lo.x, lo.y, hi.x, hi.y};
        }
        wf[i] = v;
    }
    __syncthreads();

    /* groups of 16 pixels of the rimmed tile, the next one on its way while this one is multiplied; a pixel outside the
     * image reads pixel 0 instead and is zeroed as bf16 */
    f32x4 raw[2][2 * STEPS];
    bool in_image[2];
    auto fetch = [&](int set, int g) {
        const int r = 16 * g + li, py = r / hx, y = ty0 + py - s.pad, x = tx0 + (r - py * hx) - s.pad;
        in_image[set] = r < pixels && y >= 0 && y < s.h && x >= 0 && x < s.w;
        const float *src = in + (in_image[set] ? ((size_t)y * s.w + x) * s.cin : 0) + 4 * lg;
#pragma unroll
        for (int i = 0; i < 2 * STEPS; i++) raw[set][i] = *reinterpret_cast<const f32x4 *>(src + 16 * i);
    };
    auto multiply = [&](int set, int g) {
        f32x4 acc[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
        for (int ks = 0; ks < STEPS; ks++) {
            const f32x4 lo = raw[set][2 * ks], hi = raw[set][2 * ks + 1];
            u32x4 b = {pack_bf16(lo[0], lo[1]), pack_bf16(lo[2], lo[3]), pack_bf16(hi[0], hi[1]), pack_bf16(hi[2], hi[3])};
            if (!in_image[set]) b = u32x4{0, 0, 0, 0};
            acc[0] = mfma(wf[ks * 128 + lane], b, acc[0]);
            acc[1] = mfma(wf[ks * 128 + 64 + lane], b, acc[1]);
        }
        /* rows 4 lg .. + 3 and 16 + 4 lg .. + 3 of this lane's pixel (the last four of 32 are padding) */
        float *dst = z + (16 * g + li) * FO_ROWS + 4 * lg;
        *reinterpret_cast<f32x4 *>(dst) = acc[0];
        if (lg < 3) *reinterpret_cast<f32x4 *>(dst + 16) = acc[1];
    };
    constexpr int W8 = FO_THREADS / 64;
    fetch(0, wave);
    for (int g = wave; g < groups; g += 2 * W8) {            /* two groups a turn: the register sets stay compile-time */
        if (g + W8 < groups) fetch(1, g + W8);
        multiply(0, g);
        if (g + 2 * W8 < groups) fetch(0, g + 2 * W8);
        if (g + W8 < groups) multiply(1, g + W8);
    }
    __syncthreads();

    const int oy = ty0 + threadIdx.x / FO_TX, ox = tx0 + threadIdx.x % FO_TX;
    if (oy >= s.oh || ox >= s.ow) return;
    const float *zp = z + (threadIdx.x / FO_TX * hx + threadIdx.x % FO_TX) * FO_ROWS;
    for (int co = 0; co < s.cout; co++) {
        float v = 0.0f;
        for (int ky = 0; ky < s.k; ky++)
            for (int kx = 0; kx < s.k; kx++) v += zp[(ky * hx + kx) * FO_ROWS + (ky * s.k + kx) * s.cout + co];
        out[((size_t)oy * s.ow + ox) * s.cout + co] = v + (bias ? bias[co] : 0.0f);
    }
}

template <int STEPS>
int launch_few_out(hipStream_t st, float *out, const float *in, const uint16_t *W, const float *bias, const ConvShape &s) {
    static bool configured = false;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_conv_few_out<STEPS>), hipFuncAttributeMaxDynamicSharedMemorySize, FO_LDS);
        if (e != hipSuccess) return (int)e;
        configured = true;
    }
    const int tiles_x = (s.ow + FO_TX - 1) / FO_TX, tiles = tiles_x * ((s.oh + FO_TY - 1) / FO_TY), per_xcd = (tiles + 7) / 8;
    hipLaunchKernelGGL(k_conv_few_out<STEPS>, dim3((unsigned)per_xcd * 8), dim3(FO_THREADS), FO_LDS, st, out, in, W, bias, s, tiles_x, tiles, per_xcd);
    return (int)hipGetLastError();
}

inline bool al16(const void *p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

extern "C" {

/* The shapes these kernels take; -2, with nothing enqueued, for any other. */
int iris_hip_conv2d_direct(void *stream, float *out, const float *in, const uint16_t *w, const float *bias, int h, int width,
                           int cin, int cout, int k, int stride, int pad_before, int oh, int ow) {
    hipStream_t st = (hipStream_t)stream;
    const ConvShape s = {h, width, cin, cout, k, stride, pad_before, oh, ow};
    if (k * k * cin <= 32 && (long)oh * ow <= (1L << 30)) {
        const int groups = (int)(((long)oh * ow + 15) / 16);
        const bool aligned = cout % 4 == 0 && al16(out);
        /* five workgroups a CU (32 KB of LDS each); a wave fetches its weights once for all its groups */
        const dim3 grid((unsigned)(groups < 1280 * FI_WAVES ? (groups + FI_WAVES - 1) / FI_WAVES : 1280), (unsigned)((cout + FI_COLS - 1) / FI_COLS));
        if (aligned) hipLaunchKernelGGL(k_conv_few_in<true>, grid, dim3(64 * FI_WAVES), 0, st, out, in, w, bias, s, groups);
        else hipLaunchKernelGGL(k_conv_few_in<false>, grid, dim3(64 * FI_WAVES), 0, st, out, in, w, bias, s, groups);
        return (int)hipGetLastError();
    }
    if (k <= FO_MAX_K && k * k * cout <= FO_ROWS && stride == 1 && (cin == 32 || cin == 64 || cin == 128) && al16(in) && al16(w))
        return cin == 32 ? launch_few_out<1>(st, out, in, w, bias, s) : cin == 64 ? launch_few_out<2>(st, out, in, w, bias, s)
                                                                               : launch_few_out<4>(st, out, in, w, bias, s);
    return -2;
}

}  // extern "C"
