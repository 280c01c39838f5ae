/*
 * Convolutions of a channels-last f32 image that need neither a patch matrix nor a bf16 copy of the image
 * (reference iris_dev.h:111-121, iris_cuda.cu:959-1016; the other shapes are in gemm_conv_gfx950.hip).
 *
 * k_conv_few_in: k * k * cin <= 32, the 3-channel input of the VAE encoder.
 * k_conv_few_out: k * k * cout <= 28, the 3-channel output of the VAE decoder.
 * k_conv_1x1: cin a multiple of 128, at most 512, cout at most 256: the VAE's skip connections.
 * k_conv_3x3: 3 x 3, stride 1, cin a multiple of 64: every other layer of the VAE but the halving ones.
 * k_conv_3x3_half: 3 x 3, stride 2, cin a multiple of 32, cout at least 128: those.
 * `route` says where each of them pays. The counts of workgroups in it, and in the launchers, are for the 256 CUs of an MI355X; on
 * another number of them only the choice would be another, not the results.
 *
 * The first two are bound by memory: one side of the product is so thin that the image on the other side is all there
 * is to move. The image is rounded to bf16 on the way into the matrix core, products are summed in f32.
 */
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

#include "iris_kernels_hip.h"
#include "write_through.h"

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
 * What bounds it is the output stream, as long as little else is done: a workgroup puts its weights and the places of the
 * patch's values together once in the LDS (a thread of the form before read 64 weights one by one and divided eight times), the
 * weights are on their way beside the first pixels, and a group that lies inside the image adds eight offsets to one address and tests
 * nothing. 3 -> 128 on 512 x 512 (134 MB out): 902 us as patches + scalar product + bias, 38.5 with every value tested and divided for, 28.4 without, 26.2
 * with the weights beside the pixels; likewise 64 x 64 7.1, 6.7, 5.2, 256 x 256 20.0, 10.1, 8.9, 300 x 300 23.4, 12.8, 11.3, 1024 x 1024 123, 108, 106,
 * 400 x 400, 3 -> 256 48.8, 36.7, 32.7, and, where the tests were few, 64 x 64, 4 -> 128 with 1 x 1 5.8, 6.5, 5.2, 128 x 128 6.7, 7.2, 6.0.
 * A lane without a patch value to read reads the image's first: beside the pixel's own values (more cache lines, read for nothing) 1 x 1, 4 -> 128 on
 * 1024 x 1024 119.0 / 115.5, 900 x 900 93.4 / 83.5, 4 -> 256 on 700 x 700 111.3 / 104.3, 16 -> 200 on 128 x 128 7.3 / 6.8; 3 x 3, 3 -> 128 the same. */
constexpr int FI_WAVES = 4, FI_COLS = 128, FI_BEYOND = 1 << 28;
/* Whole 512-byte pieces of a row are written through as they are stored, as long as the result is not larger than the Infinity Cache: us,
 * plain / through, 64 x 64, 3 -> 128 (2 MB) 4.4 / 4.3, 128 x 128 5.3 / 4.7, 180 x 180 7.1 / 5.9, 362 x 362 14.9 / 13.7, 512 x 512 30.6 / 26.2, 724 x 724 (268 MB) 55.1 /
 * 54.3, 1024 x 1024 (537 MB) 103 / 120; 3 -> 512 32 x 32 4.9 / 4.9, 100 x 100 7.8 / 6.8, 362 x 362 (268 MB) 53.0 / 48.9, 512 x 512 104 / 96. Rows that are not made of
 * such pieces lose by it (512 x 512, 3 -> 64 24.9 / 26.4, 7 -> 260 34 / 40). */
constexpr size_t FI_THROUGH_MOST = (size_t)256 << 20;
/* A wave has up to eight pieces on their way at once. Large results in wide rows, and the largest, are faster with one (PACED). us, eight / one,
 * 3 -> 1024 160 x 160 (105 MB) 23.0 / 24.4, 181 x 181 31.8 / 29.0, 256 x 256 61.8 / 50.3, 362 x 362 127 / 106; 768 181 x 181 (100 MB) 19.9 / 22.1, 256 x 256 42.0 /
 * 40.5, 300 x 300 58.0 / 55.8; 512 200 x 200 (82 MB) 16.6 / 18.3, 256 x 256 (134 MB) 27.8 / 27.7, 362 x 362 50.7 / 49.3; 256 362 x 362 (134 MB) 27.2 / 31.7, 600 x 600 73.7 /
 * 80.3; 128 420 x 420 19.3 / 22.9, 724 x 724 54.6 / 60.4, 900 x 900 (415 MB) 84.3 / 85.1, 1024 x 1024 110.6 / 103.3. */
constexpr size_t FI_EIGHT_MOST = (size_t)480 << 20, FI_EIGHT_MOST_WIDE = (size_t)120 << 20;
constexpr int FI_WIDE = 4;                                     /* tiles of 128 channels */

/* p / ow for p < 2^30: umulhi(p, magic) >> shift, magic = ceil(2^(32 + shift) / ow) with 2^shift < ow <= 2^(shift + 1); 0: ow is 1 */
struct RowOf { unsigned magic, shift; };
inline RowOf row_of(unsigned ow) {
    if (ow < 2) return {0, 0};
    unsigned shift = 0;
    while (2ull << shift < ow) shift++;
    return {(unsigned)(((1ull << (32 + shift)) + ow - 1) / ow), shift};
}

template <bool ALIGNED, bool THROUGH, bool PACED>
__global__ void __launch_bounds__(64 * FI_WAVES, 4)
k_conv_few_in(float *__restrict__ out, const float *__restrict__ in, const uint16_t *__restrict__ W, const float *__restrict__ bias,
              ConvShape s, RowOf row_of, int small, int groups) {
    __shared__ __align__(16) float lds[FI_WAVES * 16 * FI_COLS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, lg = lane >> 4;
    const int column = blockIdx.x, columns = gridDim.x, n0 = blockIdx.y * FI_COLS;
    const int row_len = s.k * s.k * s.cin, pixels = s.oh * s.ow;
    float *buf = lds + wave * 16 * FI_COLS;

    /* rows of 32 weights, zeros behind the patch, on their way beside the first group's pixels; and for patch value r its tap's row and
     * column (row FI_BEYOND: beyond the patch, never inside the image) and its offset from the patch's first value */
    uint16_t *w_lds = reinterpret_cast<uint16_t *>(lds);
    int *tap_y = reinterpret_cast<int *>(lds + FI_COLS * 16), *tap_x = tap_y + 32, *tap_off = tap_y + 64;
    if (threadIdx.x < 32) {
        const int r = threadIdx.x, tap = r / s.cin, c = r - tap * s.cin, y = tap / s.k, x = tap - y * s.k;
        tap_y[r] = r < row_len ? y : FI_BEYOND;
        tap_x[r] = x;
        tap_off[r] = r < row_len ? (y * s.w + x) * s.cin + c : 0;
    }
    uint16_t wv[FI_COLS * 32 / (64 * FI_WAVES)];
#pragma unroll
    for (int i = 0; i < FI_COLS * 32 / (64 * FI_WAVES); i++) {
        const int e = threadIdx.x + 64 * FI_WAVES * i, n = n0 + (e >> 5), j = e & 31;
        const bool there = n < s.cout && j < row_len;
        const uint16_t t = W[there ? (size_t)n * row_len + j : 0];
        wv[i] = there ? t : (uint16_t)0;
    }
    const int c = lane & 31, n = n0 + 4 * c;
    f32x4 bv;                                                  /* of the four channels this lane stores */
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const bool there = bias && n + r < s.cout;
        const float t = *(there ? bias + n + r : in);
        bv[r] = there ? t : 0.0f;
    }
    __syncthreads();
    int dy[8], dx[8], off[8];                                  /* of patch values 8 lg + j */
#pragma unroll
    for (int j = 0; j < 8; j++) { dy[j] = tap_y[8 * lg + j]; dx[j] = tap_x[8 * lg + j]; off[j] = tap_off[8 * lg + j]; }

    float v[8];
    auto fetch = [&](int g) {
        const int p = 16 * g + li;
        const int oy = row_of.magic ? (int)(__umulhi((unsigned)p, row_of.magic) >> row_of.shift) : p;
        const int y0 = oy * s.stride - s.pad, x0 = (p - oy * s.ow) * s.stride - s.pad;
        const bool whole = p < pixels && y0 >= 0 && y0 + s.k <= s.h && x0 >= 0 && x0 + s.k <= s.w;
        if (small && __all(whole)) {
            const unsigned base = (unsigned)(y0 * s.w + x0) * (unsigned)s.cin;
#pragma unroll
            for (int j = 0; j < 8; j++) {                      /* what is beyond the patch reads one place, whichever the pixel */
                const unsigned at = dy[j] == FI_BEYOND ? 0 : base + (unsigned)off[j];
                v[j] = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(in) + 4u * at);
            }
#pragma unroll
            for (int j = 0; j < 8; j++)
                if (dy[j] == FI_BEYOND) v[j] = 0.0f;
            return;
        }
        const long base = ((long)y0 * s.w + x0) * s.cin;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int y = y0 + dy[j], x = x0 + dx[j];
            const bool inside = p < pixels && (unsigned)y < (unsigned)s.h && (unsigned)x < (unsigned)s.w;
            const float t = in[inside ? base + off[j] : 0];
            v[j] = inside ? t : 0.0f;
        }
    };
    int g = column * FI_WAVES + wave;
    if (g < groups) fetch(g);
#pragma unroll
    for (int i = 0; i < FI_COLS * 32 / (64 * FI_WAVES); i++) w_lds[threadIdx.x + 64 * FI_WAVES * i] = wv[i];
    __syncthreads();
    u32x4 av[8];
#pragma unroll
    for (int a = 0; a < 8; a++) av[a] = *reinterpret_cast<const u32x4 *>(&w_lds[(16 * a + li) * 32 + 8 * lg]);
    __syncthreads();                                           /* the LDS is the waves' from here on */
    for (; g < groups; g += columns * FI_WAVES) {
        const u32x4 b = {pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7])};
        /* lane: channels 16 a + 4 lg .. + 3 of pixel li. 16-byte chunk c of pixel r in slot (c & 16) | ((c ^ r) & 15): the
         * writes (16 pixels, one chunk) and the reads (32 chunks of a pixel) both spread over all banks. A wave's own
         * region, and the LDS serves a wave's instructions in order: no barrier. */
#pragma unroll
        for (int a = 0; a < 8; a++) {
            const int chunk = 4 * a + lg;
            *reinterpret_cast<f32x4 *>(&buf[li * FI_COLS + 4 * ((chunk & 16) | ((chunk ^ li) & 15))]) = mfma(av[a], b, f32x4{0, 0, 0, 0});
        }
        if (g + columns * FI_WAVES < groups) fetch(g + columns * FI_WAVES);         /* on its way while this group is stored */
        float *first = out + (size_t)(16 * g) * s.cout + n0;    /* the same for the wave */
#pragma unroll
        for (int it = 0; it < 8; it++) {
            const int row = 2 * it + (lane >> 5);
            const f32x4 r = *reinterpret_cast<const f32x4 *>(&buf[row * FI_COLS + 4 * ((c & 16) | ((c ^ row) & 15))]) + bv;
            float *dst = first + (unsigned)(row * s.cout + 4 * c);
            if (PACED) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if (16 * g + row >= pixels) continue;
            if (ALIGNED && THROUGH) {
                if (n < s.cout) store_through(dst, r);
            } else if (ALIGNED) {
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
 * memory (a k-step's 32 channels as two 16-byte loads a lane, channels 4 lg and 16 + 4 lg, so that a load covers 64 B of
 * a pixel), and only Z passes through the LDS. A workgroup makes Z for the (32 + k - 1) x (16 + k - 1) pixels under a 32 x 16
 * tile of the output (1.2 x, the overlap comes from the L2).
 * What bounds it is the read of the image. 128 -> 3 on 1024 x 1024 (537 MB in): 1383 us as patches + 128-wide product +
 * bias, 122 us here (5.3 TB/s with the overlap). Two workgroups per CU (Z and the weights take 78 KB of LDS), so that one
 * adds while one reads. */
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

/* ---- 1 x 1 ----
 *
 * A product of the image with a small matrix. A workgroup keeps the weights of 128 output channels in the LDS for as long as
 * it lives, as A operands in the order the waves read them, and its sixteen waves walk blocks of 16 pixels: a wave fetches
 * its pixels straight into registers as f32 (two 16-byte loads per k-step, so that a load covers 64 B of a pixel), rounds
 * them there and multiplies them with all 128 channels, one LDS read per product. While a group of 128 input channels
 * is multiplied the next one, or the next block's first, is on its way. Nothing is shared between waves but the weights:
 * no barrier.
 * What bounds it is the image and the result: 512 x 512 pixels, 256 -> 128 channels 76 + 65 us as a bf16 copy and an implicit
 * product, 85 here (402 MB; eight waves that take 32 pixels each, half an LDS read per product, 2 more; pixels of images of 192 MB
 * and more read with the streaming hint 80, but other channels 10 - 20 % slower: 512 x 512, 256 -> 64 66 / 69, 202 MB, 384 -> 100 62 / 78,
 * and 256 -> 256, where two workgroups read every pixel, 116 / 141). With more than two
 * tiles of channels the image is read once for each (512 -> 1536 over 16384 pixels: 84 us against 61), so those go through a
 * copy (gemm_conv_gfx950.hip), as do few pixels of many channels (one_by_one_us). */
constexpr int C1_N = 128, C1_MAX_CIN = 512, C1_WAVES = 16, C1_OUT = 512;   /* output channels of a workgroup; f32 of LDS per wave for its stores */

__global__ void __launch_bounds__(64 * C1_WAVES, 4)
k_conv_1x1(float *__restrict__ out, const float *__restrict__ in, const uint16_t *__restrict__ W, const float *__restrict__ bias,
           int pixels, int cin, int cout, int tiles_n, int total, int per_xcd) {
    extern __shared__ __align__(16) float lds1[];              /* C1_WAVES x C1_OUT, then the weights: [k-step][8][64 lanes] x 16 B */
    u32x4 *wf = reinterpret_cast<u32x4 *>(lds1 + C1_WAVES * C1_OUT);
    /* the channel tiles of a pixel range next to each other on an XCD: they share the image in its L2 */
    const int work = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (work >= total) return;
    const int n0 = work % tiles_n * C1_N, slot = work / tiles_n, slots = total / tiles_n;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, lg = lane >> 4;

    for (int i = threadIdx.x; i < cin / 32 * 512; i += 64 * C1_WAVES) {
        const int ks = i >> 9, n = n0 + 16 * ((i >> 6) & 7) + (i & 15), g = (i >> 4) & 3;
        u32x4 v = {0, 0, 0, 0};
        if (n < cout) {                                        /* a lane's eight channels are 4 g .. + 3 and 16 + 4 g .. + 3 */
            const uint16_t *src = W + (size_t)n * cin + 32 * ks + 4 * g;
            const uint2 lo = *reinterpret_cast<const uint2 *>(src), hi = *reinterpret_cast<const uint2 *>(src + 16);
            v = u32x4{lo.x, lo.y, hi.x, hi.y};
        }
        wf[i] = v;
    }
    __syncthreads();

    const int blocks = (pixels + 15) / 16, groups = cin / 128, stride = slots * C1_WAVES;
    float *buf = lds1 + wave * C1_OUT;
    const int c = lane & 7;
    f32x4 bias4[4];
#pragma unroll
    for (int h = 0; h < 4; h++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int n = n0 + 32 * h + 4 * c + e;
            bias4[h][e] = bias && n < cout ? bias[n] : 0.0f;
        }
    const bool chunks = cout % 4 == 0 && ((uintptr_t)out & 15) == 0;

    f32x4 raw[8];                                              /* [k-step, half] of a group of 128 channels */
    auto fetch = [&](int block, int group) {
        const int p = min(16 * block + li, pixels - 1);
        const float *src = in + (size_t)p * cin + 128 * group + 4 * lg;
#pragma unroll
        for (int i = 0; i < 8; i++) raw[i] = *reinterpret_cast<const f32x4 *>(src + 16 * i);
    };
    int block = slot * C1_WAVES + wave;
    if (block < blocks) fetch(block, 0);
    for (; block < blocks; block += stride) {
        f32x4 acc[8];
#pragma unroll
        for (int a = 0; a < 8; a++) acc[a] = f32x4{0, 0, 0, 0};
        for (int group = 0; group < groups; group++) {
            u32x4 bv[4];
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
                const f32x4 lo = raw[2 * ks], hi = raw[2 * ks + 1];
                bv[ks] = u32x4{pack_bf16(lo[0], lo[1]), pack_bf16(lo[2], lo[3]), pack_bf16(hi[0], hi[1]), pack_bf16(hi[2], hi[3])};
            }
            const bool last = group + 1 == groups;
            if (!last || block + stride < blocks) fetch(last ? block + stride : block, last ? 0 : group + 1);
#pragma unroll
            for (int ks = 0; ks < 4; ks++)
#pragma unroll
                for (int a = 0; a < 8; a++) acc[a] = mfma(wf[((4 * group + ks) * 8 + a) * 64 + lane], bv[ks], acc[a]);
        }
        /* acc[a][r]: channel n0 + 16 a + 4 lg + r of pixel 16 block + li. Through the LDS (a wave's own region), 16
         * pixels x 32 channels at a time, so that a store instruction covers eight pixels x 128 B. */
#pragma unroll
        for (int h = 0; h < 4; h++) {
#pragma unroll
            for (int a = 0; a < 2; a++) *reinterpret_cast<f32x4 *>(&buf[li * 32 + 4 * ((4 * a + lg) ^ (li & 7))]) = acc[2 * h + a];
#pragma unroll
            for (int it = 0; it < 2; it++) {
                const int row = 8 * it + (lane >> 3), p = 16 * block + row, n = n0 + 32 * h + 4 * c;
                const f32x4 v = *reinterpret_cast<const f32x4 *>(&buf[row * 32 + 4 * (c ^ (row & 7))]) + bias4[h];
                if (p >= pixels) continue;
                float *dst = out + (size_t)p * cout + n;
                if (chunks) {
                    if (n < cout) *reinterpret_cast<f32x4 *>(dst) = v;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (n + e < cout) dst[e] = v[e];
                }
            }
        }
    }
}

/* workgroups per tile of channels: about one per CU in all, but no more than there are blocks of 16 x 16 pixels for */
int one_by_one_slots(int pixels, int cout) {
    const int slots = 256 / ((cout + C1_N - 1) / C1_N), most = (pixels + 16 * C1_WAVES - 1) / (16 * C1_WAVES);
    return slots < 1 ? 1 : slots < most ? slots : most;
}

int launch_1x1(hipStream_t st, float *out, const float *in, const uint16_t *W, const float *bias, int pixels, int cin, int cout) {
    static bool configured = false;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_conv_1x1), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return (int)e;
        configured = true;
    }
    const int tiles_n = (cout + C1_N - 1) / C1_N, slots = one_by_one_slots(pixels, cout);
    const int total = slots * tiles_n, per_xcd = (total + 7) / 8;
    hipLaunchKernelGGL(k_conv_1x1, dim3((unsigned)per_xcd * 8), dim3(64 * C1_WAVES), C1_WAVES * C1_OUT * 4 + cin * 256, st, out, in, W, bias, pixels,
                       cin, cout, tiles_n, total, per_xcd);
    return (int)hipGetLastError();
}

/* ---- 3 x 3 ----
 *
 * A workgroup makes 16 x 16 output pixels of 128 channels. For 64 input channels at a time, the 18 x 18 pixels under the
 * tile are read ONCE as f32, rounded and kept in the LDS; the nine taps are nine shifted views of them, so the image
 * passes from the L2 to the CU 1.27 times instead of nine, and no bf16 copy of it is made first. The weights of a (tap,
 * 64 channels) step, 128 rows of 128 B, go straight from memory into one of three LDS stages.
 *
 * Twelve waves, three per SIMD, with roles of their own, so that nobody's loads stand in the way of anybody else's:
 *  - Waves 0 - 7 multiply: 4 (rows of four pixels) x 2 (64 channels), a wave owns 64 pixels x 64 channels = 4 x 4
 *    accumulator blocks, and a step is 32 products: 16 of the first half of the step's channels, the barrier, 16 of the
 *    second half. The operands of a half are read from the LDS in the gaps between the products of the half before, one to
 *    a gap, behind its first four (a decoder stage 128 x 128, 512 -> 512, from the first gap on 860.5 us, behind four 849.5, behind six 853.5), across
 *    the barrier too: four of weights, and of a tap's four rows of pixels one where the tap before was the one above
 *    it, which the order of the taps makes two of three (all four read for every tap: 2 - 3 % more on the sizes below).
 *    They issue no load and wait for none, so a tile's stores drain under the next tile.
 *  - Waves 8 - 11 bring everything in. The image: 2592 units of 8 channels x pixel per group of 64 channels, 11 a thread,
 *    all of them in registers on their way while the group before is multiplied. One or two a step are rounded and written
 *    to the image buffer that the last group has left (the epilogue borrows it until the barrier of step 0), and
 *    requested again for the group after the next, of the next tile if there is one. The weights: those of step s + 2
 *    into the stage that the barrier of step s - 1 has set free; they have landed in front of the barrier of step s + 1.
 * A pixel takes 160 B of LDS (64 channels + 32 B): the 16 lanes that a 128-bit read serves together are eight pixels with
 * one chunk and the eight between them with the next, and with a stride of ten 16 B units, whichever pixel the
 * tap starts at, they fall into distinct bank windows; a tap's shift is an immediate offset. Weight rows are swizzled as
 * in gemm_conv_gfx950.hip. A workgroup takes 152 KB of LDS, so a CU runs one, and it is persistent.
 *
 * A tile of 512 input channels takes 44 us on however few CUs, and a round of few tiles as long as a full one. So the tiles of an XCD
 * behind its whole rounds may be cut into ranges of channel groups, dealt to its 32 CUs in equal shares (c3_share); what lies in a
 * range is a tile like any other, but leaves its sums in a workspace, and k_conv_3x3_sum adds the ranges in order. `three_ranges` says
 * where that is the faster form. A convolution under capture, which may be replayed on any stream, has no workspace and keeps its tiles whole.
 *
 * Measured against a bf16 copy of the image + implicit product that fetches every tap from the L2 (copy + product), against
 * eight waves that did everything (and stood still while a tile's stores landed), and these roles: 512 x 512 pixels, 128 -> 128
 * 30 + 118, 79, 73 us (the image and the result alone take 50 us to move), 256 -> 128 76 + 214, 129, 123, 256 -> 256 88 + 290,
 * 253, 235 us. Then the taps down the columns and the reads behind four products, on a slower chip: these roles / now, the image in the Infinity Cache,
 * 75.9 / 74.3, 137.3 / 133.3, 257.9 / 250.3 (1240 TFLOP/s, 0.87 us a step), 256 x 256, 512 -> 512 228.5 / 218.9; the image from memory 80.8 / 79.7, 140.0 / 135.6, 257.9 /
 * 251.0, 235.7 / 226.5. The first is bound by memory (matrix cores busy 43 - 45 % of its cycles), the last by the products
 * at the clock that the chip's power leaves (62 - 64 % at 1.9 - 2.0 GHz of 2.4; counters, under the profiler). Pixels and
 * weights on waves of their own (three and one) 1 % slower. */
constexpr int C3_T = 16, C3_H = C3_T + 2, C3_PIXELS = C3_H * C3_H, C3_ROW = 80, C3_IMG = C3_PIXELS * C3_ROW;   /* elements */
constexpr int C3_N = 128, C3_STAGE = C3_N * 64;
constexpr int C3_MUL = 8, C3_BRING = 4, C3_THREADS = 64 * (C3_MUL + C3_BRING);           /* waves that multiply, that bring pixels and weights */
constexpr int C3_UNITS = (C3_PIXELS * 8 + 64 * C3_BRING - 1) / (64 * C3_BRING), C3_PIECES = C3_N / 8 / C3_BRING;
constexpr int C3_BIAS = 2 * C3_IMG + 3 * C3_STAGE;             /* the bias of all output channels, f32 */
constexpr int C3_MAX_COUT = (160 * 1024 - 2 * C3_BIAS) / 4 / C3_N * C3_N;
/* units written and requested again in a step of a channel group */
__device__ constexpr int c3_first(int t) { return t < 1 ? 0 : t < 4 ? 2 * (t - 1) : t + 2; }
__device__ constexpr int c3_units(int t) { return c3_first(t + 1) - c3_first(t); }
static_assert(c3_first(9) == C3_UNITS && c3_units(0) == 0, "");
/* the tap of a step: down the columns of the 3 x 3 */
__device__ constexpr int c3_tap(int t) { return t % 3 * 3 + t / 3; }

/* Results of up to 64 MB are written through (write_through.h), larger ones stay for the operator that reads them next: us, plain /
 * through, a decoder stage 64 x 70, 512 -> 512 308.0 / 301.8, the first encoder stage 150 x 200 107.1 / 104.3, 256 x 256 144.0 / 141.9, 320 x 330 (54 MB)
 * 205.3 / 203.8, 512 x 512 (134 MB) 399.3 / 408.0; alone 256 x 256, 128 -> 128 (34 MB) 24.3 / 23.2, 128 x 250, 512 -> 512 (66 MB) 117.5 / 117.2, 256 x 256, 256 -> 256 (67
 * MB) 67.0 / 66.7, 181 x 181, 512 -> 512 137.4 / 138.5, 362 x 362, 128 -> 128 (67 MB) 53.9 / 54.2, 400 x 400 (82 MB) 58.6 / 61.5, 450 x 450 77.4 / 82.0,
 * 362 x 362, 256 -> 256 (134 MB) 143.6 / 146.7; but 1024 x 1024, 128 -> 128 (537 MB) 310.4 / 308.4. */
constexpr size_t C3_THROUGH_MOST = (size_t)64 << 20;
constexpr int C3_SLOTS = 32, C3_PART = 4096;                   /* CUs of an XCD; floats of a wave's sums */
static_assert((size_t)16 * C3_SLOTS * C3_MUL * C3_PART * 4 <= IRIS_LINEAR_PART_BYTES, "two places a workgroup");

__device__ __forceinline__ uint32_t lds_address(const uint16_t *p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)p;
}

/* What a workgroup takes of its XCD's tiles [first, ..): whole ones up to rest_first, every slots-th; and, where the last round is cut,
 * channel groups [u0, u1) of the `rest` tiles behind them, counted through those tiles, of which every taker has one at least. As
 * rest < slots, these are at most a tile's number of groups and lie in at most two tiles. */
struct C3Share { int first, rest_first, rest, takers, u0, u1; };
__host__ __device__ inline C3Share c3_share(int xcd, int slot, int slots, int total, int per_xcd, int groups, bool cut) {
    const int first = xcd * per_xcd < total ? xcd * per_xcd : total, end = first + per_xcd < total ? first + per_xcd : total;
    if (!cut) return {first, end, 0, 0, 0, 0};
    const int rest = (end - first) % slots, all = rest * groups, takers = all < slots ? all : slots;
    return {first, end - rest, rest, takers, slot < takers ? all * slot / takers : all, slot < takers ? all * (slot + 1) / takers : all};
}
/* The workgroup that has channel group `unit` of the rest: the last with all * slot / takers < unit + 1 */
__host__ __device__ inline int c3_taker(const C3Share &sh, int groups, int unit) { return ((unit + 1) * sh.takers - 1) / (sh.rest * groups); }

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"                /* M0 in a clobber list */
__global__ void __launch_bounds__(C3_THREADS, 3)
k_conv_3x3(float *__restrict__ out, const float *__restrict__ in, const uint16_t *__restrict__ W, const float *__restrict__ bias,
           ConvShape s, int tiles_x, int tiles_n, int total, int per_xcd, float *__restrict__ part, int through) {
    extern __shared__ __align__(16) uint16_t lds[];            /* image, image, weights, weights, weights, bias */
    /* an XCD takes a contiguous range of the tiles, the channel tiles of a pixel tile next to each other (they share the
     * image in its L2), dealt out to its workgroups in turn; with `part`, those of its last, incomplete round in ranges of channel groups */
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int groups = s.cin / 64, slot = blockIdx.x / 8, slots = gridDim.x / 8;
    const C3Share sh = c3_share(blockIdx.x % 8, slot, slots, total, per_xcd, groups, part != nullptr);
    /* the grid has C3_SLOTS workgroups an XCD, or one per tile of it */
    const int wholes = slot >= sh.rest_first - sh.first ? 0 : slots == C3_SLOTS ? (sh.rest_first - sh.first - slot + C3_SLOTS - 1) / C3_SLOTS : 1;
    const int units = wholes * groups + sh.u1 - sh.u0;         /* channel groups of tiles that this workgroup takes */
    if (units == 0) return;
    int p_w = sh.rest_first, p_g = 0;                          /* where its range begins */
    if (part) {
        p_w += sh.u0 / groups;
        p_g = sh.u0 % groups;
    }
    const int w_first = wholes ? sh.first + slot : p_w, g_first = wholes ? 0 : p_g;
    auto next = [&](int &w, int &g) {
        if (++g < groups) return;
        g = 0;
        if (w >= sh.rest_first) {
            w++;
        } else if ((w += slots) >= sh.rest_first) {
            w = p_w;
            g = p_g;
        }
    };
    float *bias_lds = reinterpret_cast<float *>(lds + C3_BIAS);
    for (int i = tid; i < tiles_n * C3_N; i += C3_THREADS) bias_lds[i] = bias && i < s.cout ? bias[i] : 0.0f;

    /* Every wave passes one barrier here in front and nine per channel group, in every role. */
    if (wave >= C3_MUL) {
        __builtin_amdgcn_s_setprio(3);
        const int bt = tid - 64 * C3_MUL, bw = wave - C3_MUL, px0 = bt >> 3;
        /* weights: rows 8 (C3_PIECES bw + j) .. + 7 of a stage; rows past the last channel repeat it (their results are never
         * stored). When nothing comes next the last requests are of weights that nobody uses. */
        const int row_len = 9 * s.cin;
        uint32_t woff[C3_PIECES];
        auto aim_weights = [&](int w) {
            const int n = w % tiles_n * C3_N;
#pragma unroll
            for (int j = 0; j < C3_PIECES; j++) {
                const int r = 8 * (C3_PIECES * bw + j) + (lane >> 3), row = n + r < s.cout ? n + r : s.cout - 1;
                woff[j] = ((uint32_t)row * (uint32_t)row_len + 8u * ((lane & 7) ^ ((r >> 1) & 7))) * 2u;
            }
        };
        const uint32_t stages = lds_address(lds + 2 * C3_IMG + C3_PIECES * bw * 8 * 64);
        auto request = [&](int t, int c0) {                    /* the stage of step t: t % 3 */
            const uint16_t *src = W + (size_t)c3_tap(t) * s.cin + c0;
#pragma unroll
            for (int j = 0; j < C3_PIECES; j++)
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                             ::"s"(stages + 2 * (t % 3 * C3_STAGE + 8 * j * 64)), "v"(woff[j]), "s"(src) : "memory", "m0");
        };
        /* pixels: unit u of this thread is channels 8 (bt % 8) .. + 7 of pixel bt / 8 + 32 u of the rimmed tile; a pixel
         * outside the image reads the first one and is zeroed */
        uint32_t off[C3_UNITS], inside = 0, held = 0;          /* bytes from the channel group's first value; bit u: in the image */
        int w = w_first, g = g_first, left = units;            /* where the next loads come from */
        const float *src = in + 64 * g;
        auto aim = [&]() {
            const int tile = w / tiles_n, ty = tile / tiles_x * C3_T - s.pad, tx = tile % tiles_x * C3_T - s.pad;
            int first = px0;
            asm volatile("" : "+v"(first));                    /* worked out here for every tile: kept over the loop it all spills */
            inside = 0;
#pragma unroll
            for (int u = 0; u < C3_UNITS; u++) {
                const int px = first + 8 * C3_BRING * u, py = px / C3_H, y = ty + py, x = tx + (px - py * C3_H);
                const bool ok = px < C3_PIXELS && y >= 0 && y < s.h && x >= 0 && x < s.w;
                if (ok) inside |= 1u << u;
                off[u] = ((ok ? (uint32_t)(y * s.w + x) * (uint32_t)s.cin : 0u) + 8u * (bt & 7)) * 4u;
            }
        };
        auto advance = [&]() {
            if (--left > 0) {
                const int tile = w;
                next(w, g);
                src = in + 64 * g;
                if (w != tile) aim();
            } else {                                           /* nothing comes next: the same loads, of a few cached bytes that nobody uses */
                src = in;
                inside = 0;
#pragma unroll
                for (int u = 0; u < C3_UNITS; u++) off[u] = 32u * (bt & 7);
            }
        };
        f32x4 xr[C3_UNITS][2];
        auto load = [&](int u) {
            const char *p = reinterpret_cast<const char *>(src) + off[u];
            xr[u][0] = *reinterpret_cast<const f32x4 *>(p);
            xr[u][1] = *reinterpret_cast<const f32x4 *>(p + 16);
        };
        auto put = [&](int img, int u) {
            const f32x4 lo = xr[u][0], hi = xr[u][1];
            u32x4 v = {pack_bf16(lo[0], lo[1]), pack_bf16(lo[2], lo[3]), pack_bf16(hi[0], hi[1]), pack_bf16(hi[2], hi[3])};
            if (!(held >> u & 1)) v = u32x4{0, 0, 0, 0};
            if (u + 1 < C3_UNITS || px0 < C3_PIXELS - 8 * C3_BRING * (C3_UNITS - 1))
                *reinterpret_cast<u32x4 *>(&lds[img + (px0 + 8 * C3_BRING * u) * C3_ROW + 8 * (bt & 7)]) = v;
        };
        aim_weights(w);
        request(0, 64 * g);
        request(1, 64 * g);
        aim();
#pragma unroll
        for (int u = 0; u < C3_UNITS; u++) load(u);
        held = inside;
        advance();
#pragma unroll
        for (int u = 0; u < C3_UNITS; u++) {
            put(0, u);
            load(u);
            __builtin_amdgcn_sched_barrier(0);
        }
        /* everything older than the loads just issued is there */
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * C3_UNITS) : "memory");
        int cw = w_first, cg = g_first;                        /* what is multiplied meanwhile */
        for (int img = 0, unit = 0; unit < units; unit++, img = C3_IMG - img) {
            const bool more = unit + 1 < units;
            int nw = cw, ng = cg;
            next(nw, ng);
            held = inside;
            advance();
#pragma unroll
            for (int t = 0; t < 9; t++) {
                if (t == 7 && more && nw != cw) aim_weights(nw);
                if (t < 7) request(t + 2, 64 * cg);
                else request(t - 7, more ? 64 * ng : 0);
#pragma unroll
                for (int u = c3_first(t); u < c3_first(t + 1); u++) {
                    put(C3_IMG - img, u);
                    load(u);
                }
                __builtin_amdgcn_sched_barrier(0);
                /* newer than the weights of step t + 1: two loads a unit in the step that requested them and in this
                 * one, and the weights of step t + 2 */
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier"
                             ::"n"(2 * (c3_units(t > 0 ? t - 1 : 8) + c3_units(t)) + C3_PIECES) : "memory");
                __builtin_amdgcn_sched_barrier(0);
            }
            cw = nw;
            cg = ng;
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       /* no load into the LDS is left when it is given up */
        return;
    }

    const int li = lane & 15, lg = lane >> 4, wm = wave & 3, wn = wave >> 2;
    /* [16 channels][row of 16 pixels]. The products are asm statements: left to itself the compiler gives a product's result
     * other registers than its summand, and 168 are not enough for that. It does not know then when a result is there
     * and when a summand must be: `settle` stands between the products and any other use of acc. */
    f32x4 acc[4][4];
    auto settle = [&]() {
        asm volatile("s_nop 15" : "+v"(acc[0][0]), "+v"(acc[0][1]), "+v"(acc[0][2]), "+v"(acc[0][3]), "+v"(acc[1][0]), "+v"(acc[1][1]),
                                  "+v"(acc[1][2]), "+v"(acc[1][3]), "+v"(acc[2][0]), "+v"(acc[2][1]), "+v"(acc[2][2]), "+v"(acc[2][3]),
                                  "+v"(acc[3][0]), "+v"(acc[3][1]), "+v"(acc[3][2]), "+v"(acc[3][3]));
    };
    auto clear = [&]() {
#pragma unroll
        for (int a = 0; a < 4; a++)
#pragma unroll
            for (int b = 0; b < 4; b++) acc[a][b] = f32x4{0, 0, 0, 0};
        settle();
    };
    u32x4 av[2][4], bv[2][4];
    int a_rd[2];
#pragma unroll
    for (int ks = 0; ks < 2; ks++) a_rd[ks] = 2 * C3_IMG + (64 * wn + li) * 64 + 8 * ((4 * ks + lg) ^ (li >> 1));
    const int b_rd = (4 * wm * C3_H + li) * C3_ROW + 8 * lg;
    /* operand i of a half of step t, in the order its products use them. Row r of pixels, counted from the wave's first in the rimmed
     * tile, is kept in bv[ks][r % 4]: three steps go down a column of taps, and of the second and third only the last row is new. */
    auto operand = [&](int img, int t, int ks, int i) {
        if (i == 0 || i > 4) {
            const int a = i == 0 ? 0 : i - 4;
            av[ks][a] = *reinterpret_cast<const u32x4 *>(&lds[a_rd[ks] + (t % 3) * C3_STAGE + 16 * a * 64]);
        } else if (t % 3 == 0 || i == 4) {
            const int r = i - 1 + t % 3;
            bv[ks][r % 4] = *reinterpret_cast<const u32x4 *>(&lds[img + b_rd + (r * C3_H + t / 3) * C3_ROW + 32 * ks]);
        }
    };
    auto products = [&](int ks, int t, int img, int next) {    /* of step t; img, next: of the operands read on the way */
#pragma unroll
        for (int i = 0; i < 16; i++) {
            asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc[i / 4][i % 4]) : "v"(av[ks][i / 4]), "v"(bv[ks][(i + t % 3) % 4]));
            if (i >= 4 && i < 12) operand(img, next, ks ^ 1, i - 4);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    /* acc[a][b][r]: channel n0 + 64 wn + 16 a + 4 lg + r of pixel (4 wm + b, li) of the tile. Through the image buffer that the
     * last group has been read from (every wave has passed the barrier behind its last reads, and the next pixels go into
     * it behind the next barrier; 4 KB per wave, a row of 16 pixels at a time), so that a store instruction covers four
     * pixels x 256 B. */
    const bool chunks = s.cout % 4 == 0 && ((uintptr_t)out & 15) == 0;
    auto epilogue = [&](int img, int w) {
        const int tile = w / tiles_n, n0 = (w - tile * tiles_n) * C3_N, ty0 = tile / tiles_x * C3_T, tx0 = tile % tiles_x * C3_T;
        float *buf = reinterpret_cast<float *>(lds + img) + wave * 1024;
        int li = lane & 15, lg = lane >> 4;
        asm volatile("" : "+v"(li), "+v"(lg));                 /* the addresses are worked out here: kept over the loop they spill */
        const int c = li, n = n0 + 64 * wn + 4 * c;
        const f32x4 bias4 = *reinterpret_cast<const f32x4 *>(bias_lds + n);
        const bool whole = chunks && ty0 + C3_T <= s.oh && tx0 + C3_T <= s.ow && n0 + C3_N <= s.cout;
#pragma unroll
        for (int b = 0; b < 4; b++) {
#pragma unroll
            for (int a = 0; a < 4; a++) *reinterpret_cast<f32x4 *>(&buf[li * 64 + 4 * ((4 * a + lg) ^ li)]) = acc[a][b];
            const int y = ty0 + 4 * wm + b;
            f32x4 v[4];
#pragma unroll
            for (int it = 0; it < 4; it++) {
                const int row = 4 * it + lg;
                v[it] = *reinterpret_cast<const f32x4 *>(&buf[row * 64 + 4 * (c ^ row)]) + bias4;
            }
            float *dst = out + ((size_t)y * s.ow + tx0 + lg) * s.cout + n;
            if (whole && through) {
#pragma unroll
                for (int it = 0; it < 4; it++) store_through(dst + (size_t)(4 * it) * s.cout, v[it]);
            } else if (whole) {
#pragma unroll
                for (int it = 0; it < 4; it++) *reinterpret_cast<f32x4 *>(dst + (size_t)(4 * it) * s.cout) = v[it];
            } else if (y < s.oh) {
#pragma unroll
                for (int it = 0; it < 4; it++) {
                    if (tx0 + 4 * it + lg >= s.ow) continue;
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (n + e < s.cout) dst[(size_t)(4 * it) * s.cout + e] = v[it][e];
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    /* the sums of a range of channel groups, as the registers hold them: 128 KB, two places a workgroup. Written through, as the next
     * kernel reads them: us, plain / through, decoder stages 32 x 32, 512 -> 512 128.0 / 125.7, 64 x 70 305.7 / 301.9, 33 x 40, 512 -> 256 148.9 / 143.7, 64 x 64,
     * 256 -> 128 129.6 / 130.0; alone 32 x 32, 512 -> 512 19.2 / 18.3, 64 x 64 31.3 / 30.3, 16 x 16 15.5 / 16.4, 64 x 64, 256 -> 256 17.5 / 18.1. */
    auto store_part = [&](int w) {
        float *dst = part + ((size_t)(2 * blockIdx.x + (w != p_w)) * C3_MUL + wave) * C3_PART;
#pragma unroll
        for (int a = 0; a < 4; a++)
#pragma unroll
            for (int b = 0; b < 4; b++) store_through(dst + ((4 * a + b) * 64 + lane) * 4, acc[a][b]);
    };

    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    clear();
#pragma unroll
    for (int i = 0; i < 8; i++) operand(0, 0, 0, i);
    int w = w_first, g = g_first;
    bool from_start = g == 0;
    for (int img = 0, unit = 0; unit < units; unit++, img = C3_IMG - img) {
#pragma unroll
        for (int t = 0; t < 9; t++) {
            products(0, t, img, t);
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            products(1, t, t < 8 ? img : C3_IMG - img, t < 8 ? t + 1 : 0);
        }
        int nw = w, ng = g;
        next(nw, ng);
        if (nw != w || unit + 1 == units) {
            settle();
            if (from_start && g + 1 == groups) epilogue(img, w);
            else store_part(w);
            clear();
            from_start = ng == 0;
        }
        w = nw;
        g = ng;
    }
}
#pragma clang diagnostic pop

/* Adds the ranges of the tiles that were cut, in the order of their channels, and the bias. A workgroup takes what one wave of
 * k_conv_3x3 left of a tile, on the XCD that made it. */
__global__ void __launch_bounds__(256)
k_conv_3x3_sum(float *__restrict__ out, const float *__restrict__ part, const float *__restrict__ bias, ConvShape s, int tiles_x, int tiles_n, int total,
               int per_xcd) {
    const int xcd = blockIdx.x % 8, wave = blockIdx.x / 8 % C3_MUL, t = blockIdx.x / 8 / C3_MUL, groups = s.cin / 64;
    const C3Share sh = c3_share(xcd, 0, C3_SLOTS, total, per_xcd, groups, true);
    if (t >= sh.rest) return;
    const int first = c3_taker(sh, groups, t * groups), ranges = c3_taker(sh, groups, (t + 1) * groups - 1) - first + 1, w = sh.rest_first + t;
    if (ranges == 1) return;                                   /* one workgroup took all of it, and has stored it */
    const int place = c3_share(xcd, first, C3_SLOTS, total, per_xcd, groups, true).u0 < t * groups;
    const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4, ab0 = threadIdx.x >> 6;
    const auto at = [&](int r) {
        return part + ((size_t)(2 * (8 * (first + r) + xcd) + (r == 0 ? place : 0)) * C3_MUL + wave) * C3_PART + threadIdx.x * 4;
    };
    f32x4 v[4];
    const float *p = at(0);
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = *reinterpret_cast<const f32x4 *>(p + i * 1024);
#pragma unroll 2
    for (int r = 1; r < ranges; r++) {
        p = at(r);
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] += *reinterpret_cast<const f32x4 *>(p + i * 1024);
    }
    const int tile = w / tiles_n, n0 = (w - tile * tiles_n) * C3_N + 64 * (wave >> 2) + 4 * lg;
    const int x = tile % tiles_x * C3_T + li, y0 = tile / tiles_x * C3_T + 4 * (wave & 3);
    const bool chunks = s.cout % 4 == 0 && ((uintptr_t)out & 15) == 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int n = n0 + 16 * i, y = y0 + ab0;               /* block 4 i + ab0 of the wave's: channels 16 i, pixel row ab0 */
        if (x >= s.ow || y >= s.oh || n >= s.cout) continue;
        float *dst = out + ((size_t)y * s.ow + x) * s.cout + n;
        if (chunks) {
            if (bias) {
#pragma unroll
                for (int e = 0; e < 4; e++) v[i][e] += bias[n + e];
            }
            *reinterpret_cast<f32x4 *>(dst) = v[i];
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n + e < s.cout) dst[e] = v[i][e] + (bias ? bias[n + e] : 0.0f);
        }
    }
}

/* Whether the last round is worth cutting. It saves channel groups of 5.3 us, and costs a launch and the partial sums' way through memory,
 * 128 KB a piece and about 0.25 us for one on each XCD. us, whole / cut: 512 -> 256 64 x 69 43.7 / 29.6, 84 x 89 44.8 / 36.6, 100 x 107 46.7 / 44.1,
 * 124 x 133 47.9 / 52.0, 174 x 187 (one tile over a round on most XCDs) 91.3 / 71.3, 194 x 207 99.3 / 93.2, 217 x 233 101.9 / 112.9; 512 -> 512
 * 122 x 131 92.5 / 75.1, 174 x 187 143.3 / 122.5; 256 -> 256 64 x 69 26.3 / 20.1, 82 x 87 27.2 / 30.0, 242 x 259 81.1 / 74.6; 256 -> 128 249 x 267
 * 57.6 / 46.5; 128 -> 128 169 x 181 19.0 / 32.3, 249 x 267 37.0 / 34.3, which the rule leaves whole. */
bool three_ranges(const ConvShape &s, int per_xcd) {
    const int groups = s.cin / 64, rest = per_xcd % C3_SLOTS, units = (rest * groups + C3_SLOTS - 1) / C3_SLOTS;
    if (rest == 0) return false;
    const int pieces = rest * groups < C3_SLOTS ? rest * groups : C3_SLOTS + rest;
    return 5.3f * (float)(groups - units) > 6.0f + 0.25f * (float)pieces;
}

int launch_3x3(hipStream_t st, float *part, float *out, const float *in, const uint16_t *W, const float *bias, const ConvShape &s) {
    static bool configured = false;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_conv_3x3), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return (int)e;
        configured = true;
    }
    const int tiles_x = (s.ow + C3_T - 1) / C3_T, tiles_n = (s.cout + C3_N - 1) / C3_N;
    const int total = tiles_x * ((s.oh + C3_T - 1) / C3_T) * tiles_n, per_xcd = (total + 7) / 8;
    const unsigned lds = 2 * C3_BIAS + 4 * C3_N * (unsigned)tiles_n;
    /* one workgroup per CU (its LDS): 32 per XCD, each walking the XCD's tiles */
    if (!three_ranges(s, per_xcd)) part = nullptr;
    hipLaunchKernelGGL(k_conv_3x3, dim3((unsigned)(part || per_xcd >= C3_SLOTS ? C3_SLOTS : per_xcd) * 8), dim3(C3_THREADS), lds, st, out, in, W, bias, s,
                       tiles_x, tiles_n, total, per_xcd, part, (size_t)s.oh * s.ow * s.cout * 4 <= C3_THROUGH_MOST);
    int rest = 0;                                              /* of the XCD that has most of it: the last one may have fewer tiles */
    for (int x = 0; part && x < 8; x++) {
        const int r = c3_share(x, 0, C3_SLOTS, total, per_xcd, s.cin / 64, true).rest;
        rest = r > rest ? r : rest;
    }
    if (part)
        hipLaunchKernelGGL(k_conv_3x3_sum, dim3((unsigned)rest * 8 * C3_MUL), dim3(256), 0, st, out, part, bias, s, tiles_x, tiles_n,
                           total, per_xcd);
    return (int)hipGetLastError();
}

/* ---- 3 x 3 with stride 2 ----
 *
 * The halving layers of the VAE encoder, in the manner of k_conv_3x3: 8 x 16 output pixels of 128 channels, the 17 x 33 pixels
 * under them read once as f32 and kept in the LDS as bf16, 32 channels at a time in two buffers. A step is a row of three
 * taps: eight waves, 4 (two rows of pixels) x 2 (64 channels), take 24 products each, the operands of a tap read in the gaps
 * between the products of the one before; the barrier stands in front of the last tap's products. Behind the barrier of
 * step s its weights' stage (two of 24 KB) is free and wave 11 requests those of step s + 2. Waves 8 - 10 keep the pixels of
 * the next group but one on their way, four units of 8 channels x pixel a step.
 * A pixel takes 80 B: neighbouring outputs' pixels are 160 B apart, as in k_conv_3x3. 16 B chunk c of weight row r sits
 * in slot c ^ {0, 2, 3, 1}[r / 4 % 4] of its 64 B: the 16 lanes that a 128-bit read serves together, rows 0 - 3 and
 * 12 - 15 with one chunk and 4 - 11 with its neighbour, then hit distinct bank windows.
 * Bound by the image where there are few channels (512 x 512 x 128 in, 167 MB with the result: 30 us at the rate of a copy), by
 * the products otherwise. Against a bf16 copy of the image + implicit product: 512 x 512, 128 -> 128 63 -> 42 us, 1024 x 1024
 * 304 -> 164, 128 x 128 30 -> 12, 256 x 256, 256 -> 256 77 -> 28, 128 x 128, 512 -> 512 119 -> 42, 256 x 256 143 -> 113. Pixels
 * straight into registers under every tap instead of a shared tile (nine reads of 2.25 outputs' pixels each): 55 us for the
 * first, 92 for 256 -> 256: a CU takes in 50 - 65 KB/us of what is not in its XCD's L2.
 * Results are written through (write_through.h) at every size: us, plain / through, image from memory, 512 x 512, 128 -> 128 (34 MB) 45.7 / 44.6, 640 x 640 75.5 /
 * 75.8, 724 x 724 (67 MB) 93.6 / 94.1, 800 x 800 102.3 / 103.6, 900 x 900 (104 MB) 136.4 / 136.1, 1024 x 1024 (134 MB) 163.3 / 163.0, 256 -> 256 362 x 362 (34 MB) 87.5 / 86.6,
 * 512 x 512 (67 MB) 128.2 / 128.0, 724 x 724 (134 MB) 282.6 / 279.7, 512 -> 512 256 x 256 (34 MB) 110.4 / 109.1, 400 x 400 (82 MB) 325.6 / 322.1, 512 x 512 440.4 / 437.6. */
constexpr int H3_TY = 8, H3_TX = 16, H3_HY = 2 * H3_TY + 1, H3_HX = 2 * H3_TX + 1, H3_PIXELS = H3_HY * H3_HX, H3_C = 32, H3_ROW = 40;
constexpr int H3_IMG = H3_PIXELS * H3_ROW, H3_TAP = C3_N * H3_C, H3_STAGE = 3 * H3_TAP;      /* elements */
constexpr int H3_BRING = 3, H3_THREADS = 64 * (C3_MUL + H3_BRING + 1), H3_PIECES = H3_STAGE / 512;
constexpr int H3_UNITS = (H3_PIXELS * 4 + 64 * H3_BRING - 1) / (64 * H3_BRING);
constexpr int H3_OUT = 2 * H3_IMG + 2 * H3_STAGE, H3_BIAS = H3_OUT + C3_MUL * 1024;          /* 2 KB per wave for its stores; bias */
constexpr int H3_MAX_COUT = (160 * 1024 - 2 * H3_BIAS) / 4 / C3_N * C3_N;
static_assert(H3_UNITS == 12 && H3_PIECES == 24 && H3_IMG % 8 == 0, "four units a step");

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"                /* M0 in a clobber list */
__global__ void __launch_bounds__(H3_THREADS, 3)
k_conv_3x3_half(float *__restrict__ out, const float *__restrict__ in, const uint16_t *__restrict__ W, const float *__restrict__ bias,
                ConvShape s, int tiles_x, int tiles_n, int total, int per_xcd) {
    extern __shared__ __align__(16) uint16_t lds[];            /* image, image, weights, weights, outputs, bias */
    const int xcd_end = min((int)(blockIdx.x % 8 + 1) * per_xcd, total), stride = gridDim.x / 8;
    int work = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (work >= xcd_end) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int groups = s.cin / H3_C;
    float *bias_lds = reinterpret_cast<float *>(lds + H3_BIAS);
    for (int i = tid; i < tiles_n * C3_N; i += H3_THREADS) bias_lds[i] = bias && i < s.cout ? bias[i] : 0.0f;

    /* Every wave passes one barrier here in front and three per channel group, in every role. */
    if (wave >= C3_MUL + H3_BRING) {
        /* weights: request j brings rows 16 (j % 8) .. + 15 of tap j / 8 of the row; rows past the last channel repeat it
         * (their results are never stored). When nothing comes next the last requests are of weights that nobody uses. */
        __builtin_amdgcn_s_setprio(3);
        uint32_t off[8];
        auto aim = [&](int w) {
            const int n = w % tiles_n * C3_N;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int r = 16 * j + (lane >> 2), row = n + r < s.cout ? n + r : s.cout - 1, k4 = (r >> 2) & 3;
                const int swizzle = ((k4 << 1) ^ (k4 >> 1) * 3) & 3;
                off[j] = ((uint32_t)row * (uint32_t)(9 * s.cin) + 8u * ((lane & 3) ^ swizzle)) * 2u;
            }
        };
        const uint32_t stages = lds_address(lds + 2 * H3_IMG);
        auto request = [&](int row, int c0, int stage) {
#pragma unroll
            for (int j = 0; j < H3_PIECES; j++)
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                             ::"s"(stages + 2 * (stage * H3_STAGE + j * 512)), "v"(off[j % 8]), "s"(W + (size_t)(3 * row + j / 8) * s.cin + c0)
                             : "memory", "m0");
        };
        aim(work);
        request(0, 0, 0);
        request(1, 0, 1);
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(H3_PIECES) : "memory");
        for (int g = 0, stage = 0; work < xcd_end;) {
            const bool last = g + 1 == groups;
#pragma unroll
            for (int t = 0; t < 3; t++) {
                asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");      /* those of the next step are there */
                if (t == 1 && last && work + stride < xcd_end) aim(work + stride);
                if (t == 0) request(2, H3_C * g, stage);
                else request(t - 1, last ? 0 : H3_C * (g + 1), stage);
                stage ^= 1;
            }
            g = last ? 0 : g + 1;
            if (last) work += stride;
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       /* no load into the LDS is left when it is given up */
        return;
    }
    if (wave >= C3_MUL) {
        /* pixels: unit u of this thread is channels 8 (bt % 4) .. + 7 of pixel bt / 4 + 48 u of the rimmed tile; a pixel
         * outside the image reads the first one and is zeroed */
        __builtin_amdgcn_s_setprio(3);
        const int bt = tid - 64 * C3_MUL, px0 = bt >> 2;
        uint32_t off[H3_UNITS], inside = 0, held = 0;          /* bytes from the channel group's first value; bit u: in the image */
        int w = work, g = 0;                                   /* where the next loads come from */
        const float *src = in;
        auto aim = [&]() {
            const int tile = w / tiles_n, ty = tile / tiles_x * (2 * H3_TY) - s.pad, tx = tile % tiles_x * (2 * H3_TX) - s.pad;
            int first = px0;
            asm volatile("" : "+v"(first));                    /* worked out here for every tile: kept over the loop it all spills */
            inside = 0;
#pragma unroll
            for (int u = 0; u < H3_UNITS; u++) {
                const int px = first + 16 * H3_BRING * u, py = px / H3_HX, y = ty + py, x = tx + (px - py * H3_HX);
                const bool ok = px < H3_PIXELS && y >= 0 && y < s.h && x >= 0 && x < s.w;
                if (ok) inside |= 1u << u;
                off[u] = ((ok ? (uint32_t)(y * s.w + x) * (uint32_t)s.cin : 0u) + 8u * (bt & 3)) * 4u;
            }
        };
        auto advance = [&]() {
            if (g + 1 < groups) {
                g++;
                src += H3_C;
            } else {
                src = in;
                g = 0;
                w += stride;
                if (w < xcd_end) {
                    aim();
                } else {                                       /* nothing comes next: the same loads, of a few cached bytes that nobody uses */
                    inside = 0;
#pragma unroll
                    for (int u = 0; u < H3_UNITS; u++) off[u] = 32u * (bt & 3);
                }
            }
        };
        f32x4 xr[H3_UNITS][2];
        auto load = [&](int u) {
            const char *p = reinterpret_cast<const char *>(src) + off[u];
            xr[u][0] = *reinterpret_cast<const f32x4 *>(p);
            xr[u][1] = *reinterpret_cast<const f32x4 *>(p + 16);
        };
        auto put = [&](int img, int u) {
            const f32x4 lo = xr[u][0], hi = xr[u][1];
            u32x4 v = {pack_bf16(lo[0], lo[1]), pack_bf16(lo[2], lo[3]), pack_bf16(hi[0], hi[1]), pack_bf16(hi[2], hi[3])};
            if (!(held >> u & 1)) v = u32x4{0, 0, 0, 0};
            if (u + 1 < H3_UNITS || px0 < H3_PIXELS - 16 * H3_BRING * (H3_UNITS - 1))
                *reinterpret_cast<u32x4 *>(&lds[img + (px0 + 16 * H3_BRING * u) * H3_ROW + 8 * (bt & 3)]) = v;
        };
        aim();
#pragma unroll
        for (int u = 0; u < H3_UNITS; u++) load(u);
        held = inside;
        advance();
#pragma unroll
        for (int u = 0; u < H3_UNITS; u++) {
            put(0, u);
            load(u);
            __builtin_amdgcn_sched_barrier(0);
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        for (int img = 0, gg = 0; work < xcd_end; img = H3_IMG - img) {
            held = inside;
            advance();
#pragma unroll
            for (int t = 0; t < 3; t++) {
#pragma unroll
                for (int u = 4 * t; u < 4 * t + 4; u++) {
                    put(H3_IMG - img, u);
                    load(u);
                }
                __builtin_amdgcn_sched_barrier(0);
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            }
            if (++gg == groups) { gg = 0; work += stride; }
        }
        return;
    }

    const int li = lane & 15, lg = lane >> 4, wm = wave & 3, wn = wave >> 2;
    f32x4 acc[4][2];                                           /* [16 channels][row of 16 pixels] */
    auto clear = [&]() {
#pragma unroll
        for (int a = 0; a < 4; a++)
#pragma unroll
            for (int b = 0; b < 2; b++) acc[a][b] = f32x4{0, 0, 0, 0};
    };
    u32x4 av[2][4], bv[2][2];
    const int k4 = li >> 2, a_rd = 2 * H3_IMG + (64 * wn + li) * H3_C + 8 * (lg ^ (((k4 << 1) ^ (k4 >> 1) * 3) & 3));
    const int b_rd = (4 * wm * H3_HX + 2 * li) * H3_ROW + 8 * lg;
    /* operand i of a tap, in the order its products use them */
    auto operand = [&](int set, int img, int stage, int ky, int kx, int i) {
        if (i == 0 || i > 2) {
            const int a = i == 0 ? 0 : i - 2;
            av[set][a] = *reinterpret_cast<const u32x4 *>(&lds[a_rd + stage * H3_STAGE + kx * H3_TAP + 16 * a * H3_C]);
        } else {
            bv[set][i - 1] = *reinterpret_cast<const u32x4 *>(&lds[img + b_rd + ((2 * (i - 1) + ky) * H3_HX + kx) * H3_ROW]);
        }
    };
    auto products = [&](int set, int img, int stage, int ky, int kx) {       /* img .. kx: of the operands read on the way */
#pragma unroll
        for (int i = 0; i < 8; i++) {
            acc[i / 2][i % 2] = mfma(av[set][i / 2], bv[set][i % 2], acc[i / 2][i % 2]);
            if (i < 6) operand(set ^ 1, img, stage, ky, kx, i);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    /* acc[a][b][r]: channel n0 + 64 wn + 16 a + 4 lg + r of pixel (2 wm + b, li) of the tile. Through the LDS (2 KB, a wave's
     * own region), 16 pixels x 32 channels at a time, so that a store instruction covers eight pixels x 128 B. */
    const bool chunks = s.cout % 4 == 0 && ((uintptr_t)out & 15) == 0;
    auto epilogue = [&]() {
        const int tile = work / tiles_n, n0 = (work - tile * tiles_n) * C3_N, ty0 = tile / tiles_x * H3_TY, tx0 = tile % tiles_x * H3_TX;
        float *buf = reinterpret_cast<float *>(lds + H3_OUT) + wave * 512;
        const int c = lane & 7;
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const int y = ty0 + 2 * wm + b;
#pragma unroll
            for (int half = 0; half < 2; half++) {
#pragma unroll
                for (int a = 0; a < 2; a++) *reinterpret_cast<f32x4 *>(&buf[li * 32 + 4 * ((4 * a + lg) ^ (li & 7))]) = acc[2 * half + a][b];
                const int n = n0 + 64 * wn + 32 * half + 4 * c;
                const f32x4 bias4 = *reinterpret_cast<const f32x4 *>(bias_lds + n);
#pragma unroll
                for (int it = 0; it < 2; it++) {
                    const int row = 8 * it + (lane >> 3), x = tx0 + row;
                    const f32x4 v = *reinterpret_cast<const f32x4 *>(&buf[row * 32 + 4 * (c ^ (row & 7))]) + bias4;
                    if (y >= s.oh || x >= s.ow) continue;
                    float *dst = out + ((size_t)y * s.ow + x) * s.cout + n;
                    if (chunks) {
                        if (n < s.cout) store_through(dst, v);
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            if (n + e < s.cout) dst[e] = v[e];
                    }
                }
            }
        }
    };

    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int i = 0; i < 6; i++) operand(0, 0, 0, 0, 0, i);
    clear();
    /* nine taps a group, so operand sets and stages change places from one group to the next: two groups a turn */
    int img = 0, g = 0;
    auto channel_group = [&](auto odd) {
        constexpr int o = decltype(odd)::value;
#pragma unroll
        for (int t = 0; t < 3; t++) {
            const int stage = (t + o) & 1;
            products((3 * t + o) & 1, img, stage, t, 1);
            products((3 * t + 1 + o) & 1, img, stage, t, 2);
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            products((3 * t + 2 + o) & 1, t < 2 ? img : H3_IMG - img, stage ^ 1, t < 2 ? t + 1 : 0, 0);
        }
        img = H3_IMG - img;
        if (++g == groups) {
            epilogue();
            clear();
            g = 0;
            work += stride;
        }
    };
    while (work < xcd_end) {
        channel_group(std::integral_constant<int, 0>{});
        if (work >= xcd_end) break;
        channel_group(std::integral_constant<int, 1>{});
    }
}
#pragma clang diagnostic pop

int launch_3x3_half(hipStream_t st, float *out, const float *in, const uint16_t *W, const float *bias, const ConvShape &s) {
    static bool configured = false;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_conv_3x3_half), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return (int)e;
        configured = true;
    }
    const int tiles_x = (s.ow + H3_TX - 1) / H3_TX, tiles_n = (s.cout + C3_N - 1) / C3_N;
    const int total = tiles_x * ((s.oh + H3_TY - 1) / H3_TY) * tiles_n, per_xcd = (total + 7) / 8;
    const unsigned lds = 2 * H3_BIAS + 4 * C3_N * (unsigned)tiles_n;
    hipLaunchKernelGGL(k_conv_3x3_half, dim3((unsigned)(per_xcd < 32 ? per_xcd : 32) * 8), dim3(H3_THREADS), lds, st, out, in, W, bias, s, tiles_x,
                       tiles_n, total, per_xcd);
    return (int)hipGetLastError();
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
inline bool overlap(const void *a, size_t a_bytes, const void *b, size_t b_bytes) {
    return (uintptr_t)a < (uintptr_t)b + b_bytes && (uintptr_t)b < (uintptr_t)a + a_bytes;
}

/* Workgroups of k_conv_few_in per tile of channels. Four run on a CU at once, and one fetches its weights once for all its groups, so
 * 1024 in all: with 1280 512 x 512 pixels, 3 -> 64 take 18.7 us in place of 16.4, 1024 x 1024, 3 -> 128 123 in place of 103, with 1280 for each of eight tiles
 * (256 x 256, 3 -> 1024) 77 in place of 50. Of two or three tiles twice as many, within a tenth of the time either way (us, 1024 in all / twice as many, 400 x 400,
 * 3 -> 256 34.8 / 32.8, 512 x 512 52.9 / 53.2, 256 x 256 13.7 / 15.2). */
inline unsigned few_in_columns(int groups, int cout) {
    const int tiles_n = (cout + FI_COLS - 1) / FI_COLS, most = tiles_n == 1 ? 1024 : tiles_n < 4 ? 2048 / tiles_n : tiles_n < 1024 ? 1024 / tiles_n : 1;
    return groups < most * FI_WAVES ? (unsigned)(groups + FI_WAVES - 1) / FI_WAVES : (unsigned)most;
}

enum Route { OTHER, FEW_IN, FEW_OUT, ONE_BY_ONE, THREE, THREE_HALF };

/* Not where there is next to nothing to do per pixel: on large images the whole products of 16 pixels x 128 channels then take
 * longer than a thread per output (1 x 1, 1 -> 1 over 1024 x 1024 45 us / 11, 4 -> 4 over 512 x 512 17 / 12; 3 x 3, 1 -> 1 44.7 / 43;
 * from images of 8 channels and up, which are gathered in 16-byte pieces, 1 x 1, 32 -> 1 26 / 22). And not for 1 x 1 of 32 channels
 * to 128 and more, where every load of a wave touches 64 different cache lines: 32 -> 512 over 256 x 256 135 us / 86, 16 x 16
 * 11.2 / 10.4; on larger images the patches of the other side go through HBM (512 x 512 220 / 428). */
bool few_in_pays(const ConvShape &s, long out_pixels) {
    const int values = s.k * s.k * s.cin;
    if (out_pixels > 131072) return values * s.cout > 16 && !(s.cin % 8 == 0 && 8 * s.cout <= values);
    return !(s.k == 1 && s.cin == 32 && s.cout >= 128);
}

/* With 1 x 1 there are no taps to save, and a thread adds up and stores all the channels of its pixel: k_conv_1x1 or a copy are
 * faster from 5 channels on (128 -> 16 over 512 x 512 41 us against 33 in k_conv_1x1; 64 -> 28 over 128 x 128 13.5 / 10.2), with 64
 * input channels from 17 (64 -> 16 9.9 / 10.0). And where an image is not as wide as a tile, as one of width 1 that a
 * caller makes of all its pixels, most of a tile is empty: what fits two workgroups a CU is still faster so, beyond that the
 * estimates decide (a round of 512 tiles takes 2.7 us + 0.036 per input channel; 65536 x 1, 128 -> 3, 1 x 1 45 us / 12). */
bool few_out_pays(const ConvShape &s, long out_pixels, float copied_us) {
    if (s.k == 1 && s.cout > (s.cin <= 64 ? 16 : 4)) return false;
    const long tiles = (long)((s.oh + FO_TY - 1) / FO_TY) * ((s.ow + FO_TX - 1) / FO_TX);
    if (tiles <= 512 || tiles * FO_TX * FO_TY <= 2 * out_pixels) return true;
    return 3.0f + (float)((tiles + 511) / 512) * (2.7f + 0.036f * (float)s.cin) < copied_us;
}

/* About what k_conv_1x1 takes: every workgroup first brings all the weights of its channels into the LDS, 5 us per 128 input
 * channels whatever the image, so a few thousand pixels of 256 and more channels are faster through a copy. Measured, us,
 * k_conv_1x1 / copy: 256 -> 128 1000 pixels 16.7 / 13.3, 9216 17.4 / 16.0, 30000 19.1 / 21.9; 512 -> 128 4096 27.5 / 12.2, 16384
 * 28.6 / 19.2, 65536 33.8 / 52.9; 384 -> 256 1000 22.1 / 21.0, 9216 23.4 / 25.8. With 128 input channels it is always faster. */
float one_by_one_us(long pixels, int cin, int cout) {
    const float weights = 6.0f + (cout <= 64 ? 3.6f : 5.2f) * (float)(cin / 128), memory = 4.0f * (float)pixels * (float)(cin + cout) / 5.0e6f;
    const float chain = (pixels < 256 ? 0.6f : 1.0f) * weights + 1e-4f * (float)pixels;
    return chain > memory ? chain : memory;
}

inline long three_tiles(const ConvShape &s, int ty, int tx) {
    return (long)((s.oh + ty - 1) / ty) * ((s.ow + tx - 1) / tx) * ((s.cout + C3_N - 1) / C3_N);
}

/* The 3 x 3 kernels multiply whole tiles. An image of a few rows or columns fills only part of each, and once its tiles no
 * longer fit one round of the CUs a copy and a product over the pixels alone is faster: us, 1 x 4096 512 -> 512 190 / 113, 8 x 3000
 * 150 / 132, 20000 x 1 128 -> 128 70 / 30, with stride 2 172 / 68 for 256 -> 256. Where tiles are at least two thirds full
 * the copy never was; elsewhere the estimates decide. A tile takes 5.8 us per 64 channels (4.9 in a grid of one round),
 * with stride 2 2.3 per 32. */
bool three_pays(const ConvShape &s, int ty, int tx, float copied_us) {
    const long tiles = three_tiles(s, ty, tx), rounds = (tiles + 255) / 256, n_tiles = (s.cout + C3_N - 1) / C3_N;
    if (2 * tiles * ty * tx <= 3 * n_tiles * s.oh * s.ow) return true;
    const float tile_us = s.stride == 1 ? 3.0f + (rounds > 1 ? 5.8f : 4.9f) * (float)(s.cin / 64) : 1.5f + 2.3f * (float)(s.cin / H3_C);
    return 3.0f + (float)rounds * tile_us <= copied_us / 0.97f;
}

/* Which kernel a convolution takes, host arithmetic only. All of them store results while other workgroups still read the
 * image around them, so an output that shares memory with the image goes elsewhere: those routes copy the image first. */
Route route(const ConvShape &s, const void *out, const void *in, const void *w) {
    const size_t in_bytes = (size_t)s.h * s.w * s.cin * 4, out_bytes = (size_t)s.oh * s.ow * s.cout * 4;
    if (overlap(out, out_bytes, in, in_bytes)) return OTHER;
    const bool plain = s.k == 1 && s.stride == 1 && s.oh == s.h && s.ow == s.w;
    const long out_pixels = (long)s.oh * s.ow;
    if (s.k * s.k * s.cin <= 32 && out_pixels <= (1L << 30) && few_in_pays(s, out_pixels)) return FEW_IN;
    const float copied_us = iris_hip_conv2d_copied_us((long)s.h * s.w, out_pixels, s.cin, s.cout, s.k, plain);
    if (s.k <= FO_MAX_K && s.k * s.k * s.cout <= FO_ROWS && s.stride == 1 && (s.cin == 32 || s.cin == 64 || s.cin == 128) && al16(in) && al16(w) &&
        few_out_pays(s, out_pixels, copied_us))
        return FEW_OUT;
    if (plain && s.cin % 128 == 0 && s.cin <= C1_MAX_CIN && s.cout <= 2 * C1_N && al16(in) && ((uintptr_t)w & 7) == 0 &&
        (s.cin == 128 || one_by_one_us(out_pixels, s.cin, s.cout) < copied_us))
        return ONE_BY_ONE;
    /* a thread's byte offsets into image and weights are 32-bit */
    const bool offsets = in_bytes < ((size_t)1 << 32) && (size_t)s.cout * 9 * s.cin * 2 < ((size_t)1 << 32);
    if (s.k == 3 && s.stride == 1 && s.cin % 64 == 0 && s.cout <= C3_MAX_COUT && al16(in) && al16(w) && offsets &&
        three_pays(s, C3_T, C3_T, copied_us))
        return THREE;
    if (s.k == 3 && s.stride == 2 && s.cin % H3_C == 0 && s.cout >= 128 && s.cout <= H3_MAX_COUT && al16(in) && al16(w) && offsets &&
        three_pays(s, H3_TY, H3_TX, copied_us))
        return THREE_HALF;
    return OTHER;
}

}  // namespace

extern "C" {

/* How k_conv_3x3 cuts the last round of `total` tiles of `groups` channel groups, for tests: share = first, rest_first, rest, u0 and u1 of a
 * workgroup; returns the workgroup of the XCD that has channel group `unit` of the rest (-1: it has none). */
int iris_hip_conv2d_share(int xcd, int slot, int total, int groups, int unit, int *share) {
    const C3Share sh = c3_share(xcd, slot, C3_SLOTS, total, (total + 7) / 8, groups, true);
    share[0] = sh.first; share[1] = sh.rest_first; share[2] = sh.rest; share[3] = sh.u0; share[4] = sh.u1;
    return unit < sh.rest * groups ? c3_taker(sh, groups, unit) : -1;
}

/* whether k_conv_3x3 does so for an output of this size where it has a workspace */
int iris_hip_conv2d_cut(int oh, int ow, int cin, int cout) {
    const ConvShape s = {oh, ow, cin, cout, 3, 1, 1, oh, ow};
    return three_ranges(s, (int)((three_tiles(s, C3_T, C3_T) + 7) / 8));
}

/* plan[0] = the kernel such a convolution takes: 1 k_conv_few_in, 2 k_conv_few_out, 3 k_conv_1x1, 4 k_conv_3x3, 5 k_conv_3x3_half,
 * 0 none of them; plan[1] = how many pieces of work its busiest wave (1, 3) or workgroup takes one after the other.
 * No GPU needed: the addresses are only compared. */
void iris_hip_conv2d_plan(const void *out, const void *in, const void *w, int h, int width, int cin, int cout, int k, int stride,
                          int pad_before, int pad_after, int *plan) {
    const int oh = (h + pad_before + pad_after - k) / stride + 1, ow = (width + pad_before + pad_after - k) / stride + 1;
    const ConvShape s = {h, width, cin, cout, k, stride, pad_before, oh, ow};
    const auto turns = [](long work, long takers) { return (int)((work + takers - 1) / takers); };
    plan[0] = route(s, out, in, w);
    plan[1] = 1;
    if (plan[0] == FEW_IN) {
        const int groups = (int)(((long)oh * ow + 15) / 16);
        plan[1] = turns(groups, (long)few_in_columns(groups, cout) * FI_WAVES);
    } else if (plan[0] == ONE_BY_ONE) {
        plan[1] = turns(((long)h * width + 15) / 16, (long)one_by_one_slots(h * width, cout) * C1_WAVES);
    } else if (plan[0] == THREE || plan[0] == THREE_HALF) {
        plan[1] = turns(plan[0] == THREE ? three_tiles(s, C3_T, C3_T) : three_tiles(s, H3_TY, H3_TX), 256);
    }
}

/* The shapes these kernels take; -2, with nothing enqueued, for any other. part: IRIS_LINEAR_PART_BYTES of private workspace, 16-byte
 * aligned, or null: no tile's input channels are then cut into ranges. */
int iris_hip_conv2d_direct(void *stream, float *part, float *out, const float *in, const uint16_t *w, const float *bias, int h, int width,
                           int cin, int cout, int k, int stride, int pad_before, int oh, int ow) {
    hipStream_t st = (hipStream_t)stream;
    const ConvShape s = {h, width, cin, cout, k, stride, pad_before, oh, ow};
    switch (route(s, out, in, w)) {
    case FEW_IN: {
        const int groups = (int)(((long)oh * ow + 15) / 16);
        const int tiles_n = (cout + FI_COLS - 1) / FI_COLS;
        const dim3 grid(few_in_columns(groups, cout), (unsigned)tiles_n);
        const RowOf rows = row_of((unsigned)ow);
        const int small = (size_t)h * width * cin * 4 < (size_t)1 << 31;          /* 32-bit byte offsets */
        const size_t out_bytes = (size_t)oh * ow * cout * 4;
        const bool through = cout % FI_COLS == 0 && out_bytes <= FI_THROUGH_MOST;
        auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(64 * FI_WAVES), 0, st, out, in, w, bias, s, rows, small, groups); };
        const bool paced = out_bytes > (tiles_n >= FI_WIDE ? FI_EIGHT_MOST_WIDE : FI_EIGHT_MOST);
        if (cout % 4 || !al16(out)) go(k_conv_few_in<false, false, false>);
        else if (paced) go(through ? k_conv_few_in<true, true, true> : k_conv_few_in<true, false, true>);
        else go(through ? k_conv_few_in<true, true, false> : k_conv_few_in<true, false, false>);
        return (int)hipGetLastError();
    }
    case FEW_OUT:
        return cin == 32 ? launch_few_out<1>(st, out, in, w, bias, s) : cin == 64 ? launch_few_out<2>(st, out, in, w, bias, s)
                                                                               : launch_few_out<4>(st, out, in, w, bias, s);
    case ONE_BY_ONE: return launch_1x1(st, out, in, w, bias, h * width, cin, cout);
    case THREE: return launch_3x3(st, part, out, in, w, bias, s);
    case THREE_HALF: return launch_3x3_half(st, out, in, w, bias, s);
    default: return -2;
    }
}

}  // extern "C"
