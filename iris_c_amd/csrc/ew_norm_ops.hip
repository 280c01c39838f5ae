/*
 * Elementwise and normalisation operators of the device API for gfx950
 * (reference iris_dev.h:45-107, 123-129; kernels iris_cuda.cu:271-400, 943-946,
 * 1018-1087). All of them are HBM-bound: one pass over the data with 16-byte
 * accesses per lane where the pointers and sizes allow it, a scalar form of
 * the same kernel otherwise.
 *
 * Row normalisations use one workgroup per row, a wave where rows are many and
 * short (row_route), and keep the row in registers between the statistics and
 * the write (rows up to 4096 floats; longer rows are read again, from cache).
 * Statistics follow the reference: LayerNorm takes the mean first and the
 * variance about it. Group norm of a large image is one launch that keeps
 * what it can of the image on the chip between the statistics and the write.
 * Of others it takes the statistics in ONE pass over the image (coalesced
 * per-pixel reads, per-workgroup partial moments of every group, merged in
 * double by a small second kernel) and normalises in a second pass. Moments
 * and statistics live in a scratch buffer the caller of the launcher provides.
 */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "iris_kernels_hip.h"
#include "write_through.h"

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

namespace {

constexpr int EW_THREADS = 256;
constexpr int ROW_THREADS = 256;

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    f32x2 p = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(p, bf16x2));
}
__device__ __forceinline__ uint16_t to_bf16(float v) { return (uint16_t)(pack_bf16(v, 0.0f) & 0xffffu); }
__device__ __forceinline__ float bf_lo(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bf_hi(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }
__device__ __forceinline__ float silu(float v) { return v / (1.0f + __expf(-v)); }

/* Add, residual, SwiGLU and row norms store their results through the L2s (write_through.h), while other rows are still read. What counts is the
 * operator and the one that reads its result behind it: us, plain / written through, residual + LayerNorm 16 - 400 rows of 2560 and 3072
 * the same (8.1 - 8.5), 1000 x 3072 11.9 / 10.2, 2115 20.8 / 19.9, 4608 39.4 / 38.3, 12800 (157 MB) 117.7 / 117.4, 12000 x 4096 155.6 / 151.7; LayerNorm + a product of
 * it 16 and 64 rows the same, 100 x 3072 17.3 / 17.1, 400 23.1 / 22.8, 1000 30.4 / 29.5, 4608 85.7 / 84.8, 12800 234.6 / 234.9; SwiGLU + a product 16 x 9728 the same,
 * 64 rows 19.5 / 19.3, 512 39.6 / 39.2, 4608 x 9216 201.3 / 200.4, 12800 544 / 538; add + group norm of 8 MB 17.3 / 17.2, 134 MB 106.7 / 105.8, 537 MB 518 / 513.
 * None of 40 such pairs from 0.1 to 537 MB was slower by more than 0.4 %, so there is no bound on either side. rms_norm_residual and add_bias, called again and
 * again on the same rows, were slower for it (12800 x 3072 76 / 86, 16384 x 512 7.7 / 10.4) and store plainly; with a reader behind them they were not timed. */
inline unsigned blocks_for(size_t n, int per_block) { return (unsigned)((n + per_block - 1) / per_block); }

/* ---------------------------------------------------------------- elementwise */

enum EwOp { OP_SILU, OP_ADD, OP_ADD_ROW, OP_MULADD_ROW, OP_FILL_ROW };

/* x[i] = f(x[i], a[i] or row[i % dim]); VEC = floats per thread (4: all pointers 16-byte
 * aligned and n, dim multiples of 4; 1 otherwise). */
template <int OP, int VEC>
__global__ void __launch_bounds__(EW_THREADS)
k_ew(float *__restrict__ x, const float *__restrict__ a, const float *__restrict__ row, int dim, size_t n) {
    const size_t i = ((size_t)blockIdx.x * EW_THREADS + threadIdx.x) * VEC;
    if (i >= n) return;
    float xv[VEC], av[VEC], rv[VEC];
    if (VEC == 4) {
        if (OP != OP_FILL_ROW) *reinterpret_cast<float4 *>(xv) = *reinterpret_cast<const float4 *>(x + i);
        if (OP == OP_ADD || OP == OP_MULADD_ROW) *reinterpret_cast<float4 *>(av) = *reinterpret_cast<const float4 *>(a + i);
        if (OP == OP_ADD_ROW || OP == OP_MULADD_ROW || OP == OP_FILL_ROW)
            *reinterpret_cast<float4 *>(rv) = *reinterpret_cast<const float4 *>(row + i % dim);
    } else {
        if (OP != OP_FILL_ROW) xv[0] = x[i];
        if (OP == OP_ADD || OP == OP_MULADD_ROW) av[0] = a[i];
        if (OP == OP_ADD_ROW || OP == OP_MULADD_ROW || OP == OP_FILL_ROW) rv[0] = row[i % dim];
    }
#pragma unroll
    for (int j = 0; j < VEC; j++) {
        if (OP == OP_SILU) xv[j] = silu(xv[j]);
        if (OP == OP_ADD) xv[j] += av[j];
        if (OP == OP_ADD_ROW) xv[j] += rv[j];
        if (OP == OP_MULADD_ROW) xv[j] = fmaf(rv[j], av[j], xv[j]);
        if (OP == OP_FILL_ROW) xv[j] = rv[j];
    }
    if (VEC == 4 && (OP == OP_ADD || OP == OP_MULADD_ROW)) store_through(x + i, *reinterpret_cast<f32x4 *>(xv));
    else if (VEC == 4) *reinterpret_cast<float4 *>(x + i) = *reinterpret_cast<float4 *>(xv);
    else x[i] = xv[0];
}

inline bool al16(const void *p) { return p == nullptr || ((uintptr_t)p & 15) == 0; }

template <int OP>
int launch_ew(hipStream_t st, float *x, const float *a, const float *row, int dim, size_t n) {
    if (!n) return 0;
    const bool vec = al16(x) && al16(a) && al16(row) && n % 4 == 0 && (dim <= 0 || dim % 4 == 0);
    if (vec) hipLaunchKernelGGL((k_ew<OP, 4>), dim3(blocks_for(n, EW_THREADS * 4)), dim3(EW_THREADS), 0, st, x, a, row, dim > 0 ? dim : 4, n);
    else hipLaunchKernelGGL((k_ew<OP, 1>), dim3(blocks_for(n, EW_THREADS)), dim3(EW_THREADS), 0, st, x, a, row, dim > 0 ? dim : 1, n);
    return (int)hipGetLastError();
}

/* Stored plainly: written through, a product that reads the rows next loses more than the store gains. us, plain / written through, with
 * a product of 512 columns behind it 4096 x 512 13.2 / 15.1, 2048 x 1536 20.1 / 23.7, 4096 x 1536 21.5 / 23.9, 8192 x 1536 28.9 / 30.6; as the copy in
 * front of a 1 x 1 convolution 512 -> 512 over 4096 pixels 14.3 / 16.6, 512 -> 1536 over 7200 32.4 / 36.0. The VAE's attention block over 32 x 32
 * positions 67.8 / 67.5, 128 x 128 560 / 559. */
template <int VEC>
__global__ void __launch_bounds__(EW_THREADS)
k_f32_to_bf16(uint16_t *__restrict__ dst, const float *__restrict__ src, size_t n) {
    const size_t i = ((size_t)blockIdx.x * EW_THREADS + threadIdx.x) * VEC;
    if (i >= n) return;
    if (VEC == 8) {
        const float4 a = *reinterpret_cast<const float4 *>(src + i), b = *reinterpret_cast<const float4 *>(src + i + 4);
        *reinterpret_cast<uint4 *>(dst + i) = make_uint4(pack_bf16(a.x, a.y), pack_bf16(a.z, a.w), pack_bf16(b.x, b.y), pack_bf16(b.z, b.w));
    } else {
        dst[i] = to_bf16(src[i]);
    }
}

/* out[r, c] = silu(gate[r, c]) * up[r, c] on bf16 rows with strides */
template <int VEC>
__global__ void __launch_bounds__(EW_THREADS)
k_swiglu(uint16_t *__restrict__ out, int ldo, const uint16_t *__restrict__ gate, const uint16_t *__restrict__ up,
         int ldi, int cols, size_t n) {
    const size_t i = ((size_t)blockIdx.x * EW_THREADS + threadIdx.x) * VEC;
    if (i >= n) return;
    const size_t r = i / cols, c = i % cols;
    if (VEC == 8) {
        const uint4 g = *reinterpret_cast<const uint4 *>(gate + r * ldi + c), u = *reinterpret_cast<const uint4 *>(up + r * ldi + c);
        const uint32_t gw[4] = {g.x, g.y, g.z, g.w}, uw[4] = {u.x, u.y, u.z, u.w};
        uint32_t o[4];
#pragma unroll
        for (int j = 0; j < 4; j++) o[j] = pack_bf16(silu(bf_lo(gw[j])) * bf_lo(uw[j]), silu(bf_hi(gw[j])) * bf_hi(uw[j]));
        store_through(out + r * ldo + c, u32x4{o[0], o[1], o[2], o[3]});
    } else {
        const float g = bf_lo(gate[r * ldi + c]);
        out[r * ldo + c] = to_bf16(silu(g) * bf_lo(up[r * ldi + c]));
    }
}

/* nearest-neighbour 2x upsampling of a channels-last image: a thread reads the VEC channels under an output column and
 * stores them to both output rows, so that a wave's store is one run of memory whatever the channels, and the second read
 * of a pixel comes from the cache. Bound by the stores. Against a thread per output value, and one per input value with
 * four stores (runs of VEC channels: slow where they are all of a pixel), us: 512 x 512 x 4 5.0, 6.0, now 4.75; x 8 7.9, 9.3,
 * 7.4; 256 x 256 x 12 4.35, 5.0, 4.1; 512 x 512 x 128 132, 120, 110; 1024 x 1024 x 128 516, 476, 437 (6.1 TB/s). */
template <int VEC>
__global__ void __launch_bounds__(EW_THREADS)
k_upsample2x(float *__restrict__ out, const float *__restrict__ in, int w, int c, size_t n) {
    const size_t i = (size_t)blockIdx.x * EW_THREADS + threadIdx.x;              /* which VEC channels of a row pair of outputs */
    if (i >= n) return;
    const unsigned per_pixel = (unsigned)c / VEC;
    const size_t per_row = (size_t)2 * w * per_pixel;
    size_t y, r, x;
    if (n >> 32 == 0) {                                        /* 32-bit divisions where they do */
        y = (unsigned)i / (unsigned)per_row;
        r = (unsigned)i - (unsigned)y * (unsigned)per_row;
        x = (unsigned)r / per_pixel;
    } else {
        y = i / per_row;
        r = i - y * per_row;
        x = r / per_pixel;
    }
    const float *src = in + (y * w + x / 2) * c + (r - x * per_pixel) * VEC;
    float *dst = out + (2 * y * per_row + r) * VEC;
    if (VEC == 4) {
        const float4 v = *reinterpret_cast<const float4 *>(src);
        *reinterpret_cast<float4 *>(dst) = v;
        *reinterpret_cast<float4 *>(dst + per_row * VEC) = v;
    } else {
        const float v = *src;
        dst[0] = v;
        dst[per_row] = v;
    }
}

/* ---------------------------------------------------------------- row normalisations */

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

__device__ __forceinline__ float block_sum(float v, float *sh) {
    v = wave_sum(v);
    const int wave = threadIdx.x >> 6;
    __syncthreads();                                  /* sh may still be read from the previous reduction */
    if ((threadIdx.x & 63) == 0) sh[wave] = v;
    __syncthreads();
    return sh[0] + sh[1] + sh[2] + sh[3];
}

enum NormKind { LAYER_NORM_MOD, RMS_NORM_MOD, RMS_NORM_RESIDUAL };
/* TPR threads per row: a workgroup of 256, or a wave. VECS > 0: dim % 4 == 0, dim <= 4 * TPR * VECS, 16-byte aligned rows -> the
 * row stays in registers between the statistics and the write; EARLY: and everything the write needs is requested
 * before the first sum is waited for. VECS = 0: the row is read again. p0/p1 are (shift, scale) for LayerNorm,
 * (w, scale) for RMSNorm, (w, gate) for the residual form; out_bf is unused by the latter. */
template <int KIND, int TPR, int VECS, bool EARLY>
__global__ void __launch_bounds__(ROW_THREADS)
k_row_norm(uint16_t *__restrict__ out_bf, float *__restrict__ xres, const float *__restrict__ src,
           const float *__restrict__ p0, const float *__restrict__ p1, int rows, int dim, float eps, unsigned grid_x) {
    __shared__ float sh[4];
    const unsigned row = (blockIdx.y * grid_x + blockIdx.x) * (ROW_THREADS / TPR) + threadIdx.x / TPR;
    if (row >= (unsigned)rows) return;                                  /* the same for all threads of a row */
    const int tid = threadIdx.x % TPR;
    auto row_sum = [&](float v) { return TPR == 64 ? wave_sum(v) : block_sum(v, sh); };
    const size_t row_off = (size_t)row * dim;
    const float *xr = src + row_off;
    const int nvec = dim >> 2;
    constexpr bool CACHE = VECS > 0;
    constexpr int N = CACHE ? VECS : 1;
    float4 keep[N], pa[N], pb[N], res[N];
    const float *pa_src = KIND == LAYER_NORM_MOD ? p1 : p0, *pb_src = KIND == LAYER_NORM_MOD ? p0 : p1;   /* scale | w, shift | scale | gate */

    float s = 0.0f;
    if (CACHE) {
#pragma unroll
        for (int j = 0; j < VECS; j++) {
            const int v = tid + j * TPR;
            keep[j] = v < nvec ? *reinterpret_cast<const float4 *>(xr + 4 * v) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
        if (EARLY) {
#pragma unroll
            for (int j = 0; j < VECS; j++) {
                const int v = tid + j * TPR;
                pa[j] = pb[j] = res[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if (v < nvec) {
                    if (pa_src) pa[j] = *reinterpret_cast<const float4 *>(pa_src + 4 * v);
                    if (pb_src) pb[j] = *reinterpret_cast<const float4 *>(pb_src + 4 * v);
                    if (KIND == RMS_NORM_RESIDUAL) res[j] = *reinterpret_cast<const float4 *>(xres + row_off + 4 * v);
                }
            }
        }
#pragma unroll
        for (int j = 0; j < VECS; j++)
            s += KIND == LAYER_NORM_MOD ? (keep[j].x + keep[j].y) + (keep[j].z + keep[j].w)
                                        : (keep[j].x * keep[j].x + keep[j].y * keep[j].y) + (keep[j].z * keep[j].z + keep[j].w * keep[j].w);
    } else {
        for (int i = tid; i < dim; i += TPR) s += KIND == LAYER_NORM_MOD ? xr[i] : xr[i] * xr[i];
    }
    s = row_sum(s);
    float mean = 0.0f, inv;
    if (KIND == LAYER_NORM_MOD) {
        mean = s / (float)dim;
        float v = 0.0f;
        if (CACHE) {
#pragma unroll
            for (int j = 0; j < VECS; j++)
                if (tid + j * TPR < nvec) {
                    const float a = keep[j].x - mean, b = keep[j].y - mean, c = keep[j].z - mean, d = keep[j].w - mean;
                    v += (a * a + b * b) + (c * c + d * d);
                }
        } else {
            for (int i = tid; i < dim; i += TPR) { const float d = xr[i] - mean; v += d * d; }
        }
        inv = 1.0f / sqrtf(row_sum(v) / (float)dim + eps);
    } else {
        inv = 1.0f / sqrtf(s / (float)dim + eps);
    }

    if (CACHE) {
#pragma unroll
        for (int j = 0; j < VECS; j++) {
            const int v = tid + j * TPR;
            if (v >= nvec) continue;
            if (!EARLY) {                                       /* without a branch: an absent operand reads the row instead */
                pa[j] = *reinterpret_cast<const float4 *>((pa_src ? pa_src : xr) + 4 * v);
                pb[j] = *reinterpret_cast<const float4 *>((pb_src ? pb_src : xr) + 4 * v);
                if (KIND == RMS_NORM_RESIDUAL) res[j] = *reinterpret_cast<const float4 *>(xres + row_off + 4 * v);
            }
            const float xin[4] = {keep[j].x, keep[j].y, keep[j].z, keep[j].w};
            const float av[4] = {pa[j].x, pa[j].y, pa[j].z, pa[j].w}, bv[4] = {pb[j].x, pb[j].y, pb[j].z, pb[j].w};
            float r[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (KIND == LAYER_NORM_MOD) {
                    float n = (xin[e] - mean) * inv;
                    if (p1) n *= 1.0f + av[e];
                    if (p0) n += bv[e];
                    r[e] = n;
                } else {
                    float t = xin[e] * inv * av[e];
                    if (KIND == RMS_NORM_MOD) { if (p1) t *= 1.0f + bv[e]; }
                    else t *= p1 ? tanhf(bv[e]) : 1.0f;
                    r[e] = t;
                }
            }
            if (KIND == RMS_NORM_RESIDUAL) {
                const float4 t = res[j];
                *reinterpret_cast<float4 *>(xres + row_off + 4 * v) = make_float4(t.x + r[0], t.y + r[1], t.z + r[2], t.w + r[3]);
            } else {
                store_through(out_bf + row_off + 4 * v, u32x2{pack_bf16(r[0], r[1]), pack_bf16(r[2], r[3])});
            }
        }
    } else {
        for (int i = tid; i < dim; i += TPR) {
            float r;
            if (KIND == LAYER_NORM_MOD) {
                r = (xr[i] - mean) * inv;
                if (p1) r *= 1.0f + p1[i];
                if (p0) r += p0[i];
            } else {
                r = xr[i] * inv * p0[i];
                if (KIND == RMS_NORM_MOD) { if (p1) r *= 1.0f + p1[i]; }
                else r *= p1 ? tanhf(p1[i]) : 1.0f;
            }
            if (KIND == RMS_NORM_RESIDUAL) xres[row_off + i] += r;
            else out_bf[row_off + i] = to_bf16(r);
        }
    }
}

enum RowRoute { ROW_WORKGROUP, ROW_WORKGROUP_REREAD, ROW_WAVE, ROW_WAVE_2048, ROW_WAVE_4096, ROW_WAVE_REREAD };

/* A workgroup per row until the chip is full of them (1280 - 1536 rows at a time), then a wave per row as long as a row is short
 * enough for one: many rows pay for two barriers each what few rows gain from short chains. us, workgroup / wave:
 *   LayerNorm  1000 x 1024 4.05 / 4.05, 1800 x 1024 4.97 / 4.07, 3000 x 1536 7.1 / 5.7, 3000 x 2048 7.8 / 6.9, 3000 x 2560 9.3 / 9.7;
 *   RMSNorm    3000 x 1024 5.1 / 3.8, 12800 x 512 12.4 / 6.4, 3000 x 2048 6.2 / 5.8, 3000 x 2560 7.6 / 9.4;
 *   residual   1500 x 512 4.7 / 4.0, 12800 x 1152 34.4 / 28.7, 3000 x 1536 12.1 / 11.7, 12800 x 2048 48.2 / 47.7, 2300 x 2048 11.2 / 13.1.
 * Tens of thousands of longer LayerNorm rows (they come from HBM) are 5 - 10 % faster in waves again: 60000 x 4096 290 / 265. */
RowRoute row_route(int kind, int rows, int dim, bool aligned) {
    const bool far = kind == LAYER_NORM_MOD && rows >= 32768;
    if (!aligned || dim % 4 || dim > 4096) return (dim <= 1024 && rows >= 2048) || far ? ROW_WAVE_REREAD : ROW_WORKGROUP_REREAD;
    if (rows > 1280 && dim <= 1024) return ROW_WAVE;
    if (rows > 1280 && dim <= (kind == RMS_NORM_RESIDUAL ? 1536 : 2048)) return ROW_WAVE_2048;
    return far ? ROW_WAVE_4096 : ROW_WORKGROUP;
}

template <int KIND>
int launch_row_norm(hipStream_t st, uint16_t *out_bf, float *xres, const float *src, const float *p0,
                    const float *p1, int rows, int dim, float eps) {
    if (rows <= 0 || dim <= 0) return 0;
    const RowRoute route = row_route(KIND, rows, dim, al16(src) && al16(xres) && al16(p0) && al16(p1) && ((uintptr_t)out_bf & 7) == 0);
    const unsigned blocks = route >= ROW_WAVE ? ((unsigned)rows + ROW_THREADS / 64 - 1) / (ROW_THREADS / 64) : (unsigned)rows;
    /* a grid dimension holds less than 2^32 threads */
    const unsigned gx = blocks < 1u << 20 ? blocks : 1u << 20;
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(gx, (blocks + gx - 1) / gx), dim3(ROW_THREADS), 0, st, out_bf, xres, src, p0, p1, rows, dim, eps, gx);
    };
    switch (route) {
    case ROW_WORKGROUP: go(k_row_norm<KIND, ROW_THREADS, 4, true>); break;
    case ROW_WORKGROUP_REREAD: go(k_row_norm<KIND, ROW_THREADS, 0, false>); break;
    case ROW_WAVE: go(k_row_norm<KIND, 64, 4, true>); break;
    /* with the residual's rows too there are not enough registers to ask for everything early */
    case ROW_WAVE_2048: go(k_row_norm<KIND, 64, 8, KIND != RMS_NORM_RESIDUAL>); break;
    case ROW_WAVE_4096: go(k_row_norm<LAYER_NORM_MOD, 64, 16, false>); break;
    case ROW_WAVE_REREAD: go(k_row_norm<KIND, 64, 0, false>); break;
    }
    return (int)hipGetLastError();
}

/* ---------------------------------------------------------------- group norm
 *
 * Large images as one launch (k_gn_resident below); else two passes over the image, one for the statistics, one that normalises.
 *
 * Statistics in ONE pass: a thread sums (x - K) and (x - K)^2 over its share of a group, K being
 * the first value it reads. K is a sample of the data, so the sums stay of the size of the
 * spread and the cancellation that plain sum / sum-of-squares formulas suffer does not arise.
 * Each thread's (count, mean, M2) is then merged with the others' by the pairwise update of the
 * parallel variance algorithm: inside the workgroup in f32, across workgroups in double.
 * (The reference reads the image twice for the statistics, mean first and then the squared
 * deviations, iris_cuda.cu:1069-1074; the merged single pass gives the same moments to f32
 * rounding.) */

constexpr int GN_MAX_BLOCKS = 1024;      /* partial moments per group */

struct Moments { float n, mean, m2; };

__device__ __forceinline__ void merge(Moments &a, const Moments b) {
    if (b.n == 0.0f) return;
    const float n = a.n + b.n, d = b.mean - a.mean;
    a.mean += d * (b.n / n);
    a.m2 += b.m2 + d * d * (a.n * b.n / n);
    a.n = n;
}

/* from sums shifted by k */
__device__ __forceinline__ Moments from_shifted(float n, float k, float s, float ss) {
    Moments m = {n, 0.0f, 0.0f};
    if (n > 0.0f) { m.mean = k + s / n; m.m2 = fmaxf(ss - s * s / n, 0.0f); }
    return m;
}

/* part[(g * nblocks + b)] = moments of group g over the pixels of block b. Coalesced form: needs
 * c % 4 == 0, cg % 4 == 0 and (c / 4) dividing 256; a thread keeps one quad of channels (inside
 * one group), the workgroup walks 256 / (c / 4) pixels per step with 16-byte loads, eight of them in flight per thread:
 * 512 x 512 x 256 63 -> 49 us, 1024 x 1024 x 128 115 -> 101 (5.3 TB/s). */
__global__ void __launch_bounds__(ROW_THREADS)
k_gn_moments_quads(Moments *__restrict__ part, const float *__restrict__ in, int hw, int c, int cg, int per_block) {
    __shared__ Moments sh[ROW_THREADS];
    const int quads = c >> 2, ppi = ROW_THREADS / quads;      /* pixels per iteration */
    const int q = threadIdx.x % quads, sub = threadIdx.x / quads;
    const int start = blockIdx.x * per_block, end = min(start + per_block, hw);
    float n = 0.0f, k = 0.0f, s = 0.0f, ss = 0.0f;
    int p = start + sub;
    if (p < end) k = in[(size_t)p * c + 4 * q];
    auto take = [&](const float4 v) {
        const float a0 = v.x - k, a1 = v.y - k, a2 = v.z - k, a3 = v.w - k;
        s += (a0 + a1) + (a2 + a3);
        ss += (a0 * a0 + a1 * a1) + (a2 * a2 + a3 * a3);
        n += 4.0f;
    };
    const size_t step = (size_t)ppi * c;
    const float *src = in + (size_t)p * c + 4 * q;
    for (; p + 7 * ppi < end; p += 8 * ppi, src += 8 * step) {
        float4 v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = *reinterpret_cast<const float4 *>(src + i * step);
#pragma unroll
        for (int i = 0; i < 8; i++) take(v[i]);
    }
    for (; p < end; p += ppi, src += step) take(*reinterpret_cast<const float4 *>(src));
    sh[threadIdx.x] = from_shifted(n, k, s, ss);
    __syncthreads();
    const int groups = c / cg, qpg = cg >> 2;
    if ((int)threadIdx.x < groups) {
        Moments t = {0.0f, 0.0f, 0.0f};
        for (int sb = 0; sb < ppi; sb++)
            for (int j = 0; j < qpg; j++) merge(t, sh[sb * quads + threadIdx.x * qpg + j]);
        part[(size_t)threadIdx.x * gridDim.x + blockIdx.x] = t;
    }
}

/* Any shape: one workgroup per (group, block), scalar strided reads. */
__global__ void __launch_bounds__(ROW_THREADS)
k_gn_moments_any(Moments *__restrict__ part, const float *__restrict__ in, int hw, int c, int cg) {
    __shared__ Moments sh[ROW_THREADS];
    const int g = blockIdx.x, b = blockIdx.y;
    const size_t total = (size_t)hw * cg;
    const size_t per_block = (total + gridDim.y - 1) / gridDim.y;
    const size_t start = (size_t)b * per_block, end = start + per_block < total ? start + per_block : total;
    float n = 0.0f, k = 0.0f, s = 0.0f, ss = 0.0f;
    for (size_t i = start + threadIdx.x; i < end; i += ROW_THREADS) {
        const float v = in[(i / cg) * c + (size_t)g * cg + i % cg];
        if (n == 0.0f) k = v;
        const float a = v - k;
        s += a; ss += a * a; n += 1.0f;
    }
    sh[threadIdx.x] = from_shifted(n, k, s, ss);
    __syncthreads();
    for (int half = ROW_THREADS / 2; half > 0; half >>= 1) {
        if ((int)threadIdx.x < half) merge(sh[threadIdx.x], sh[threadIdx.x + half]);
        __syncthreads();
    }
    if (threadIdx.x == 0) part[(size_t)g * gridDim.y + b] = sh[0];
}

/* stats[g] = mean, stats[groups + g] = 1 / sqrt(var + eps) from the workgroups' partial moments, in double, one
 * workgroup per group: the mean is the count-weighted mean of the partial means, the sum of squared deviations is
 * the sum of the partial ones plus count x (partial mean - mean)^2 -- the same combination as the pairwise
 * merge, written so that it takes two sums over the partials and a single division. */
__device__ __forceinline__ double wave_sum64(double v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

/* one workgroup of 256 threads per group; a thread holds up to GN_MAX_BLOCKS / 256 partials, loaded together */
__device__ __forceinline__ double block_sum64(double v, double *sh) {
    v = wave_sum64(v);
    __syncthreads();                                   /* sh may still be read from the previous call */
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    return (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

__global__ void __launch_bounds__(256)
k_gn_finish(float *__restrict__ stats, const Moments *__restrict__ part, int groups, int nblocks, float eps) {
    __shared__ double sh[4];
    constexpr int PER = GN_MAX_BLOCKS / 256;
    const int g = blockIdx.x;
    Moments m[PER];
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int b = threadIdx.x + 256 * i;
        m[i] = b < nblocks ? part[(size_t)g * nblocks + b] : Moments{0.0f, 0.0f, 0.0f};
    }
    double n = 0.0, weighted = 0.0;
#pragma unroll
    for (int i = 0; i < PER; i++) { n += (double)m[i].n; weighted += (double)m[i].n * (double)m[i].mean; }
    n = block_sum64(n, sh);
    const double mean = n > 0.0 ? block_sum64(weighted, sh) / n : 0.0;
    double m2 = 0.0;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const double d = (double)m[i].mean - mean;
        m2 += (double)m[i].m2 + (double)m[i].n * d * d;
    }
    m2 = block_sum64(m2, sh);
    if (threadIdx.x == 0) {
        stats[g] = (float)mean;
        stats[groups + g] = (float)(1.0 / sqrt((n > 0.0 ? m2 / n : 0.0) + (double)eps));
    }
}

/* out = (x - mean[g]) * rstd[g] * gamma[ch] + beta[ch], optionally through SiLU. VEC = 4: a thread's four
 * channels are one aligned quad, which lies inside one group (c % 4 == 0 and cg % 4 == 0) or, when
 * cg % 4 != 0, is looked up channel by channel. */
template <int VEC>
__global__ void __launch_bounds__(EW_THREADS)
k_gn_normalize(float *__restrict__ out, const float *__restrict__ in, const float *__restrict__ stats,
               const float *__restrict__ gamma, const float *__restrict__ beta, int c, int cg, int groups,
               int do_silu, size_t n) {
    const size_t i = ((size_t)blockIdx.x * EW_THREADS + threadIdx.x) * VEC;
    if (i >= n) return;
    const int ch0 = (int)(i % (size_t)c);
    float v[VEC], ga[VEC], be[VEC];
    if (VEC == 4) {
        *reinterpret_cast<float4 *>(v) = *reinterpret_cast<const float4 *>(in + i);
        *reinterpret_cast<float4 *>(ga) = *reinterpret_cast<const float4 *>(gamma + ch0);
        *reinterpret_cast<float4 *>(be) = *reinterpret_cast<const float4 *>(beta + ch0);
    } else {
        v[0] = in[i]; ga[0] = gamma[ch0]; be[0] = beta[ch0];
    }
    const bool one_group = VEC == 1 || cg % 4 == 0;
    const int g0 = ch0 / cg;
    const float mean0 = stats[g0], rstd0 = stats[groups + g0];
#pragma unroll
    for (int j = 0; j < VEC; j++) {
        float mean = mean0, rstd = rstd0;
        if (!one_group) { const int g = (ch0 + j) / cg; mean = stats[g]; rstd = stats[groups + g]; }
        const float y = (v[j] - mean) * rstd * ga[j] + be[j];
        v[j] = do_silu ? silu(y) : y;
    }
    if (VEC == 4) *reinterpret_cast<float4 *>(out + i) = *reinterpret_cast<float4 *>(v);
    else out[i] = v[0];
}

/* ---- the whole norm as one launch, from 10 MB on ----
 *
 * One workgroup per CU: each reads its share of the image once, keeps as much of it as its registers and LDS hold (KEEP steps of
 * 8 KB: 138 MB in all), leaves the moments of its share, waits for the image's statistics, and writes the share normalised; only
 * what it could not keep is read a second time, the newest first, a part of which the Infinity Cache still holds. Step i of
 * workgroup b is step 256 i + b of the image, so that the chip streams through one run of memory at any time (a run of memory per
 * workgroup: 512 x 512 x 256 146 us, this way 143). Stores carry the streaming hint: they leave the L2 as they are issued and
 * not at the end of the kernel (143 -> 114 us, 1024 x 1024 x 128 278 -> 247).
 * Bound by the memory in both directions (134 MB read in 20 us), 5 - 6 us between the last value read and the first written, and
 * the launch. Against statistics, their sum and normalising as three launches, f32 image from memory, us:
 * 16384 x 512 26.7 -> 20.1, 65536 x 256 45 -> 30, 384 x 384 x 128 50 -> 33, 512 x 512 x 128 82 -> 51, 512 x 512 x 256 155 -> 108,
 * 700 x 700 x 128 146 -> 101, 1024 x 1024 x 128 294 -> 235. The line is where an image that the operator in front has left in the
 * Infinity Cache is as fast either way (from memory / cached, three launches -> one): 512 channels, 8.5 MB 13.8 -> 13.5 / 12.7 -> 13.4,
 * 9.5 MB 14.4 -> 13.7 / 13.2 -> 13.5, 10.5 MB 14.7 -> 13.9 / 13.5 -> 13.5, 16 MB 16.6 -> 15.3 / 15.8 -> 14.5.
 *
 * Everything between workgroups is a word with the number of the launch in its high half (Tagged), so that no store has to be
 * waited for and nothing is cleared between launches: a workgroup leaves the moments of its share, merged from its threads' as in
 * the other form (with one shift for the whole workgroup it was 0.3 us less, but a share that began with a pixel 300 sigma off lost
 * 3e-5 of the variance, 2e-6 this way), workgroup g < groups
 * gathers those of group g and leaves the group's statistics, all wait for these. With fences of the memory model and every
 * workgroup gathering all groups the wait took 25 us in place of 5.
 *
 * The wait is bounded and needs no workgroup to be resident beside another: one that has waited for `patience` ticks of 10 ns
 * (another process, or work on another stream, may hold CUs) gives up its share: it notes that in the counter of arrivals and in its flag and ends. The
 * counter takes such a note only while a workgroup of its launch is missing, so the one that arrives last knows how many there are,
 * gathers all groups, as the workgroups meant to may be among them, and normalises their shares itself.
 *
 * Calls that share a scratch buffer must not overlap, and the callers rule it out. If they do they get wrong values, but neither a
 * wait without end nor anything that a later call would suffer from: what is on its way once all have arrived is looked for a
 * bounded number of times; every launch adds RES_WGS arrivals, whatever happens; nothing is taken off the counter again, the
 * last to arrive notes how far it was instead (`closed`, which only grows); and flags carry the number of the launch. So when
 * everything has ended the counter is a multiple of RES_WGS, `closed` holds its state, and no word carries the next number. */
constexpr int RES_WGS = 256, RES_THREADS = 512, RES_REG = 48, RES_LDS = 18, RES_KEEP = RES_REG + RES_LDS, RES_BATCH = 8, RES_LDS_BATCH = 6;
constexpr unsigned RES_STRIDE = RES_WGS * RES_THREADS;
constexpr int RES_LDS_BYTES = RES_LDS * RES_THREADS * 16;
constexpr int RES_MIN_GROUPS = 8, RES_MAX_GROUPS = IRIS_GN_MOST_GROUPS;        /* a group's threads are at most a wave; a wave gathers the statistics */
constexpr size_t RES_MIN_BYTES = (size_t)10 << 20;
constexpr unsigned RES_PATIENCE = 1000000, RES_LATE = 1u << 20, RES_SWEEPS = 1u << 12;         /* a second or so each */
struct Tagged { unsigned long long a, b; };                    /* two floats, each with the number of the launch in its high half */
struct ResidentSync {
    unsigned long long arrivals;                               /* of all launches; in the upper 16 bits those that gave up, modulo 2^16 */
    unsigned long long closed;                                 /* the last launch that all arrived in * 2^16 + those upper bits then */
    unsigned pad[28];
    unsigned long long gave_up[RES_WGS];                       /* the launch whose share this workgroup has given up */
    Tagged stat[RES_MAX_GROUPS], part[RES_MAX_GROUPS][RES_WGS];
};
constexpr size_t SYNC_FLOATS = sizeof(ResidentSync) / sizeof(float);

__global__ void __launch_bounds__(ROW_THREADS)
k_gn_clear(unsigned *sync) {
    for (unsigned i = threadIdx.x; i < SYNC_FLOATS; i += ROW_THREADS) sync[i] = 0u;
}

/* compute units of the current device: 256 on an MI355X that is not partitioned */
int cu_count() {
    static const int n = [] {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess) return cus;
        (void)hipGetLastError();
        return 0;
    }();
    return n;
}

template <typename T> __device__ __forceinline__ T agent_load(const T *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <typename T> __device__ __forceinline__ void agent_store(T *p, T v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

/* ONCE: what is read for the last time is read with the streaming hint, in images of RES_ONCE_BYTES and more; smaller ones may still be in the
 * Infinity Cache. us without / with: 512 x 512 x 128 (134 MB) 53.2 / 51.6, 512 x 512 x 256 115 / 108, 700 x 700 x 128 108 / 101,
 * 1024 x 1024 x 128 258 / 232; 256 x 256 x 256 (67 MB) 31.8 / 31.6, 16384 x 512 20.8 / 21.9. With the hint on what is read
 * again later too: 117, 110 and 257. */
constexpr size_t RES_ONCE_BYTES = (size_t)96 << 20;
template <bool SILU, bool ONCE>
__global__ void __launch_bounds__(RES_THREADS, 2)
k_gn_resident(f32x4 *out, const f32x4 *in, const float *__restrict__ gamma, const float *__restrict__ beta, ResidentSync *sync,
              unsigned total, int c, int cg, float eps, unsigned patience) {
    extern __shared__ f32x4 kept[];                            /* [RES_LDS][RES_THREADS] */
    __shared__ Moments sh[RES_THREADS];
    __shared__ float stat[2 * RES_MAX_GROUPS];
    __shared__ unsigned verdict, to_do, found;
    const unsigned tid = threadIdx.x, b = blockIdx.x;
    const int quads = c >> 2, q = tid % quads, groups = c / cg, group = 4 * q / cg;
    /* a step is 512 quads in a row: whole pixels, so a thread keeps its quad of channels. n: this workgroup's steps */
    const unsigned steps = (total + RES_THREADS - 1) / RES_THREADS;
    auto steps_of = [&](unsigned w) { return w < steps ? (steps - w + RES_WGS - 1) / RES_WGS : 0; };
    const unsigned n = steps_of(b), at0 = b * RES_THREADS + tid;
    auto load = [&](unsigned i) { return in[min(at0 + i * RES_STRIDE, total - 1)]; };
    auto last_load = [&](unsigned at) { return ONCE ? __builtin_nontemporal_load(in + min(at, total - 1)) : in[min(at, total - 1)]; };
    constexpr unsigned long long ARRIVALS = (1ull << 48) - 1;
    /* the number of this launch, the same in all workgroups as this one has not arrived yet; words carry 31 bits of it and a one,
     * as a new scratch is all zeros */
    const unsigned long long closed = agent_load(&sync->closed), launch = (agent_load(&sync->arrivals) & ARRIVALS) / RES_WGS + 1;
    const unsigned epoch = (unsigned)launch | 1u << 31;

    /* sums of this thread's values, shifted by its first one, a batch at a time */
    float k = 0.0f, s = 0.0f, ss = 0.0f;
    if (at0 < total) k = reinterpret_cast<const float *>(in)[(size_t)at0 * 4];
    auto take = [&](const f32x4 *v, unsigned i0, auto batch) {
        float bs = 0.0f, bss = 0.0f;
#pragma unroll
        for (int j = 0; j < batch(); j++)
            if (i0 + j < n && at0 + (i0 + j) * RES_STRIDE < total) {
                const float a0 = v[j][0] - k, a1 = v[j][1] - k, a2 = v[j][2] - k, a3 = v[j][3] - k;
                bs += (a0 + a1) + (a2 + a3);
                bss += (a0 * a0 + a1 * a1) + (a2 * a2 + a3 * a3);
            }
        s += bs;
        ss += bss;
    };
    /* what cannot be kept, two batches in flight */
    if (n > RES_KEEP) {
        const std::integral_constant<int, RES_BATCH> batch;
        unsigned i = RES_KEEP;
        for (; (n - i) % RES_BATCH; i++) { const f32x4 v = load(i); take(&v, i, std::integral_constant<int, 1>{}); }
        f32x4 v[2][RES_BATCH];
        auto fetch = [&](f32x4 *dst, unsigned at) {
#pragma unroll
            for (int j = 0; j < RES_BATCH; j++) dst[j] = load(at + j);
        };
        if (i < n) {                                           /* no request behind a branch: the wait for it would be for all */
            fetch(v[0], i);
            for (; i + 2 * RES_BATCH < n; i += 2 * RES_BATCH) {
                fetch(v[1], i + RES_BATCH);
                take(v[0], i, batch);
                fetch(v[0], i + 2 * RES_BATCH);
                take(v[1], i + RES_BATCH, batch);
            }
            if (i + RES_BATCH < n) {
                fetch(v[1], i + RES_BATCH);
                take(v[0], i, batch);
                take(v[1], i + RES_BATCH, batch);
            } else {
                take(v[0], i, batch);
            }
        }
    }
    f32x4 keep[RES_REG];
    for (int g = 0; g < RES_LDS && RES_REG + g < n; g += RES_LDS_BATCH) {
        f32x4 v[RES_LDS_BATCH];
#pragma unroll
        for (int j = 0; j < RES_LDS_BATCH; j++) v[j] = last_load(at0 + min(RES_REG + g + j, n - 1) * RES_STRIDE);
#pragma unroll
        for (int j = 0; j < RES_LDS_BATCH; j++) kept[(g + j) * RES_THREADS + tid] = v[j];
        take(v, RES_REG + g, std::integral_constant<int, RES_LDS_BATCH>{});
    }
#pragma unroll
    for (int g = 0; g < RES_REG; g += RES_BATCH)
        if (g < n)
#pragma unroll
            for (int j = 0; j < RES_BATCH; j++) keep[g + j] = last_load(at0 + min(g + j, n - 1) * RES_STRIDE);
#pragma unroll
    for (int g = 0; g < RES_REG; g += RES_BATCH)
        if (g < n) take(keep + g, g, std::integral_constant<int, RES_BATCH>{});

    /* values of a group in the share of workgroup w; the last step may be a part of one */
    auto values_of = [&](unsigned w) {
        return (float)(steps_of(w) * RES_THREADS - ((steps - 1) % RES_WGS == w ? steps * RES_THREADS - total : 0)) * (4.0f / (float)groups);
    };
    auto put = [&](Tagged *t, float x, float y) {
        agent_store(&t->a, (unsigned long long)epoch << 32 | __float_as_uint(x));
        agent_store(&t->b, (unsigned long long)epoch << 32 | __float_as_uint(y));
    };
    const f32x4 ga = *reinterpret_cast<const f32x4 *>(gamma + 4 * q), be = *reinterpret_cast<const f32x4 *>(beta + 4 * q);
    /* lanes: a power of two, at most a wave; the share's moments of group g */
    const int lanes = RES_THREADS / groups, g = tid / lanes, l = tid % lanes;
    const unsigned mine = n > 0 && at0 + (n - 1) * RES_STRIDE >= total ? n - 1 : n;            /* the last step may be a part of one */
    sh[tid] = from_shifted(4.0f * (float)mine, k, s, ss);
    __syncthreads();
    {
        const int qpg = cg >> 2;
        Moments t = sh[l / qpg * quads + g * qpg + l % qpg];
        for (int off = lanes / 2; off > 0; off >>= 1) merge(t, Moments{__shfl_xor(t.n, off, 64), __shfl_xor(t.mean, off, 64), __shfl_xor(t.m2, off, 64)});
        if (l == 0) put(&sync->part[g][b], t.mean, t.m2);
    }
    /* The first wave waits for the workgroup. */
    unsigned quitters = 0;
    if (tid < 64) {
        unsigned long long before = 0;
        if (tid == 0) before = __hip_atomic_fetch_add(&sync->arrivals, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned long long t0 = wall_clock64();
        /* until the entry is this launch's in all lanes; false: this workgroup has given up its share */
        auto wait = [&](const Tagged *t, bool wanted, auto &x, auto &y) {
            constexpr int N = sizeof(x) / sizeof(float);
            for (unsigned late = 0; late < RES_LATE;) {
                unsigned long long va[N], vb[N];
#pragma unroll
                for (int i = 0; i < N; i++) {
                    va[i] = vb[i] = 0;
                    if (wanted) { va[i] = agent_load(&t[64 * i].a); vb[i] = agent_load(&t[64 * i].b); }
                }
                bool here = true;
#pragma unroll
                for (int i = 0; i < N; i++) {
                    x[i] = __uint_as_float((unsigned)va[i]);
                    y[i] = __uint_as_float((unsigned)vb[i]);
                    here = here && (unsigned)(va[i] >> 32) == epoch && (unsigned)(vb[i] >> 32) == epoch;
                }
                if (__all(!wanted || here)) return true;
                if (wall_clock64() - t0 < patience) continue;
                int gave_up = 0;
                if (tid == 0) {
                    unsigned long long seen = agent_load(&sync->arrivals);
                    while (!gave_up && (seen & ARRIVALS) / RES_WGS < launch)
                        gave_up = __hip_atomic_compare_exchange_strong(&sync->arrivals, &seen, seen + (1ull << 48), __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (gave_up) agent_store(&sync->gave_up[b], launch);
                }
                if (__any(gave_up)) return false;
                late++;                                        /* all have arrived */
            }
            return true;
        };
        /* a group's statistics from the moments of all shares, in double as k_gn_finish takes them: nothing turns what is not a
         * number into one */
        auto finish = [&](unsigned gr) {
            constexpr int N = RES_WGS / 64;
            float m[N], m2[N];
            if (!wait(&sync->part[gr][tid], true, m, m2)) return false;
            double sum = 0.0, sq = 0.0;
#pragma unroll
            for (int i = 0; i < N; i++) sum += (double)values_of(64 * i + tid) * (double)m[i];
            const double num = (double)total * (4.0 / (double)groups), mean = wave_sum64(sum) / num;
#pragma unroll
            for (int i = 0; i < N; i++) {
                const double d = (double)m[i] - mean, count = (double)values_of(64 * i + tid);
                if (count > 0.0) sq += (double)m2[i] + count * d * d;
            }
            sq = wave_sum64(sq);
            if (tid == 0) put(&sync->stat[gr], (float)mean, (float)(1.0 / sqrt(sq / num + (double)eps)));
            return true;
        };
        bool go = b >= (unsigned)groups || finish(b);
        if (go) {
            /* last to arrive: those that had given up by then (ARRIVALS is a multiple of the number less one) */
            if (tid == 0 && (before + 1) % RES_WGS == 0) {
                const unsigned long long all = ((before & ARRIVALS) + 1) / RES_WGS, gone = before >> 48;
                if (closed >> 16 == all - 1) quitters = (unsigned)(gone - closed) & 0xffffu;
                (void)__hip_atomic_fetch_max(&sync->closed, all << 16 | gone, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            quitters = __builtin_amdgcn_readfirstlane(quitters);
            if (quitters)
                for (unsigned gr = 0; gr < (unsigned)groups; gr++) (void)finish(gr);          /* theirs may be among them */
            float m[1], r[1];
            go = wait(&sync->stat[tid], tid < (unsigned)groups, m, r);
            if (tid < (unsigned)groups) { stat[tid] = m[0]; stat[RES_MAX_GROUPS + tid] = r[0]; }
        }
        if (tid == 0) { verdict = go; to_do = quitters; }
    }
    __syncthreads();
    if (!verdict) return;
    quitters = to_do;
    const float mean = stat[group], rstd = stat[RES_MAX_GROUPS + group];
    auto one = [&](float v, float g, float bt) { const float y = (v - mean) * rstd * g + bt; return SILU ? silu(y) : y; };
    auto store = [&](unsigned at, const f32x4 v) {
        if (at < total) __builtin_nontemporal_store(f32x4{one(v[0], ga[0], be[0]), one(v[1], ga[1], be[1]), one(v[2], ga[2], be[2]), one(v[3], ga[3], be[3])}, out + at);
    };
    /* steps first .. end - 1 from memory, the last first */
    auto again = [&](unsigned first, unsigned end, unsigned at) {
        if (first >= end) return;
        f32x4 v[2][RES_BATCH];
        auto fetch = [&](f32x4 *dst, unsigned from) {
#pragma unroll
            for (int j = 0; j < RES_BATCH; j++) dst[j] = last_load(at + (from + j) * RES_STRIDE);
        };
        auto put = [&](const f32x4 *src, unsigned from) {
#pragma unroll
            for (int j = RES_BATCH - 1; j >= 0; j--) store(at + (from + j) * RES_STRIDE, src[j]);
        };
        for (; (end - first) % RES_BATCH; end--) store(at + (end - 1) * RES_STRIDE, in[min(at + (end - 1) * RES_STRIDE, total - 1)]);
        if (first >= end) return;
        fetch(v[0], end - RES_BATCH);
        for (; end - first > 2 * RES_BATCH; end -= 2 * RES_BATCH) {
            fetch(v[1], end - 2 * RES_BATCH);
            put(v[0], end - RES_BATCH);
            fetch(v[0], end - 3 * RES_BATCH);
            put(v[1], end - 2 * RES_BATCH);
        }
        if (end - first > RES_BATCH) {
            fetch(v[1], first);
            put(v[0], end - RES_BATCH);
            put(v[1], first);
        } else {
            put(v[0], first);
        }
    };
#pragma unroll
    for (int g = 0; g < RES_REG; g++)
        if (g < n) store(at0 + g * RES_STRIDE, keep[g]);
    for (int g = 0; g < RES_LDS && RES_REG + g < n; g++) store(at0 + (RES_REG + g) * RES_STRIDE, kept[g * RES_THREADS + tid]);
    again(RES_KEEP, n, at0);

    if (quitters) {
        unsigned left = quitters;
        for (unsigned sweep = 0; left > 0 && sweep < RES_SWEEPS; sweep++)
            for (unsigned w = 0; w < RES_WGS; w++) {
                if (tid == 0) {
                    const unsigned f = agent_load(&sync->gave_up[w]) == launch;
                    if (f) agent_store(&sync->gave_up[w], 0ull);
                    found = f;                                 /* not verdict: other waves may not have read that yet */
                }
                __syncthreads();
                const unsigned f = found;
                __syncthreads();
                if (!f) continue;
                left--;
                again(0, steps_of(w), w * RES_THREADS + tid);
            }
    }
}

}  // namespace

extern "C" {

int iris_hip_f32_to_bf16(void *stream, uint16_t *dst, const float *src, size_t n) {
    if (!n) return 0;
    hipStream_t st = (hipStream_t)stream;
    if (al16(dst) && al16(src) && n % 8 == 0)
        hipLaunchKernelGGL(k_f32_to_bf16<8>, dim3(blocks_for(n, EW_THREADS * 8)), dim3(EW_THREADS), 0, st, dst, src, n);
    else
        hipLaunchKernelGGL(k_f32_to_bf16<1>, dim3(blocks_for(n, EW_THREADS)), dim3(EW_THREADS), 0, st, dst, src, n);
    return (int)hipGetLastError();
}

int iris_hip_silu(void *stream, float *x, size_t n) { return launch_ew<OP_SILU>((hipStream_t)stream, x, nullptr, nullptr, 0, n); }
int iris_hip_add(void *stream, float *x, const float *a, size_t n) { return launch_ew<OP_ADD>((hipStream_t)stream, x, a, nullptr, 0, n); }
int iris_hip_add_bias(void *stream, float *y, const float *bias, int rows, int cols) {
    return launch_ew<OP_ADD_ROW>((hipStream_t)stream, y, nullptr, bias, cols, (size_t)rows * cols);
}
int iris_hip_fill_rows(void *stream, float *out, const float *row, int rows, int dim) {
    return launch_ew<OP_FILL_ROW>((hipStream_t)stream, out, nullptr, row, dim, (size_t)rows * dim);
}
/* x[r, c] += gate[c] * a[r, c], gate may be NULL */
int iris_hip_residual(void *stream, float *x, const float *a, const float *gate, int rows, int dim) {
    if (!gate) return launch_ew<OP_ADD>((hipStream_t)stream, x, a, nullptr, 0, (size_t)rows * dim);
    return launch_ew<OP_MULADD_ROW>((hipStream_t)stream, x, a, gate, dim, (size_t)rows * dim);
}

int iris_hip_swiglu(void *stream, uint16_t *out, int ldo, const uint16_t *gate, const uint16_t *up, int ldi,
                    int rows, int cols) {
    const size_t n = (size_t)rows * cols;
    if (!n) return 0;
    hipStream_t st = (hipStream_t)stream;
    if (al16(out) && al16(gate) && al16(up) && cols % 8 == 0 && ldi % 8 == 0 && ldo % 8 == 0)
        hipLaunchKernelGGL(k_swiglu<8>, dim3(blocks_for(n, EW_THREADS * 8)), dim3(EW_THREADS), 0, st, out, ldo, gate, up, ldi, cols, n);
    else
        hipLaunchKernelGGL(k_swiglu<1>, dim3(blocks_for(n, EW_THREADS)), dim3(EW_THREADS), 0, st, out, ldo, gate, up, ldi, cols, n);
    return (int)hipGetLastError();
}

/* How a row norm is dealt out, host arithmetic only: kind 0 LayerNorm, 1 RMSNorm, 2 its residual form; 0 a workgroup per row that
 * keeps the row in registers, 1 one that reads it again, 2 - 4 a wave that keeps up to 1024, 2048, 4096 floats, 5 one that reads again. */
int iris_hip_row_norm_plan(int kind, int rows, int dim, int aligned) { return row_route(kind, rows, dim, aligned != 0); }

int iris_hip_upsample2x(void *stream, float *out, const float *in, int h, int width, int c) {
    const size_t n = (size_t)2 * h * width * c;                /* values of the upper output rows */
    if (!n) return 0;
    hipStream_t st = (hipStream_t)stream;
    if (al16(out) && al16(in) && c % 4 == 0)
        hipLaunchKernelGGL(k_upsample2x<4>, dim3(blocks_for(n / 4, EW_THREADS)), dim3(EW_THREADS), 0, st, out, in, width, c, n / 4);
    else
        hipLaunchKernelGGL(k_upsample2x<1>, dim3(blocks_for(n, EW_THREADS)), dim3(EW_THREADS), 0, st, out, in, width, c, n);
    return (int)hipGetLastError();
}

int iris_hip_layer_norm_mod(void *stream, uint16_t *out, const float *x, const float *shift, const float *scale,
                            int rows, int dim, float eps) {
    return launch_row_norm<LAYER_NORM_MOD>((hipStream_t)stream, out, nullptr, x, shift, scale, rows, dim, eps);
}
int iris_hip_rms_norm_mod(void *stream, uint16_t *out, const float *x, const float *w, const float *scale,
                          int rows, int dim, float eps) {
    return launch_row_norm<RMS_NORM_MOD>((hipStream_t)stream, out, nullptr, x, w, scale, rows, dim, eps);
}
int iris_hip_rms_norm_residual(void *stream, float *x, const float *a, const float *w, const float *gate,
                               int rows, int dim, float eps) {
    return launch_row_norm<RMS_NORM_RESIDUAL>((hipStream_t)stream, nullptr, x, a, w, gate, rows, dim, eps);
}

size_t iris_hip_group_norm_scratch_floats(int groups) { return SYNC_FLOATS + 3 * (size_t)groups * GN_MAX_BLOCKS + 2 * (size_t)groups; }

/* Once for a new scratch buffer: the counters of k_gn_resident, zero between calls. */
int iris_hip_group_norm_prepare_scratch(void *stream, float *scratch) {
    hipLaunchKernelGGL(k_gn_clear, dim3(1), dim3(ROW_THREADS), 0, (hipStream_t)stream, reinterpret_cast<unsigned *>(scratch));
    return (int)hipGetLastError();
}

/* What k_gn_resident takes: a thread keeps one quad of channels through all its steps, and byte offsets have 32 bits. */
static bool resident_shape(int hw, int c, int groups) {
    return hw > 0 && c > 0 && groups >= RES_MIN_GROUPS && groups <= RES_MAX_GROUPS && c % groups == 0 && c / groups % 4 == 0 &&
           RES_THREADS % (c / 4) == 0 && (size_t)hw * c / 4 < 1u << 28;
}

/* 1: an image of this size is normalised by one launch, on a device of `cus` CUs, on which its workgroups all find room at once. On
 * fewer (a partition of the device) those that do would hold their CUs until their patience ends, 10 ms at a time. Host arithmetic only. */
int iris_hip_group_norm_plan(int hw, int c, int groups, int cus) {
    return resident_shape(hw, c, groups) && (size_t)hw * c * sizeof(float) >= RES_MIN_BYTES && cus >= RES_WGS;
}

/* The norm as one launch: -2, with nothing enqueued, for what it does not take. scratch as below; patience in ticks of 10 ns. */
int iris_hip_group_norm_resident(void *stream, float *scratch, float *out, const float *in, const float *gamma, const float *beta,
                                 int hw, int c, int groups, float eps, int do_silu, unsigned patience) {
    if (!resident_shape(hw, c, groups) || !al16(in) || !al16(out) || !al16(gamma) || !al16(beta)) return -2;
    const int cg = c / groups;
    const size_t total = (size_t)hw * c / 4;
    auto go = [&](auto silu, auto once) {
        constexpr auto kernel = k_gn_resident<decltype(silu)::value, decltype(once)::value>;
        static const hipError_t configured =                   /* one for each kernel: the arguments' types tell them apart */
            hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, RES_LDS_BYTES);
        if (configured != hipSuccess) return (int)configured;
        hipLaunchKernelGGL(kernel, dim3(RES_WGS), dim3(RES_THREADS), RES_LDS_BYTES, (hipStream_t)stream, reinterpret_cast<f32x4 *>(out),
                           reinterpret_cast<const f32x4 *>(in), gamma, beta, reinterpret_cast<ResidentSync *>(scratch), (unsigned)total, c, cg, eps,
                           patience);
        return (int)hipGetLastError();
    };
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    if (total * 16 >= RES_ONCE_BYTES) return do_silu ? go(yes, yes) : go(no, yes);
    return do_silu ? go(yes, no) : go(no, no);
}

/* scratch: iris_hip_group_norm_scratch_floats(groups) floats of device memory, prepared once. Behind the counters every slot a
 * call reads (partial moments [group][workgroup], statistics [2][group]) is written by that call first. */
int iris_hip_group_norm(void *stream, float *scratch, float *out, const float *in, const float *gamma,
                        const float *beta, int hw, int c, int groups, float eps, int do_silu) {
    if (hw <= 0 || c <= 0) return 0;
    if (iris_hip_group_norm_plan(hw, c, groups, cu_count())) {
        const int e = iris_hip_group_norm_resident(stream, scratch, out, in, gamma, beta, hw, c, groups, eps, do_silu, RES_PATIENCE);
        if (e != -2) return e;
    }
    hipStream_t st = (hipStream_t)stream;
    Moments *part = reinterpret_cast<Moments *>(scratch + SYNC_FLOATS);
    float *stats = scratch + SYNC_FLOATS + 3 * (size_t)groups * GN_MAX_BLOCKS;
    const int cg = c / groups;
    const bool quads_form = c % 4 == 0 && cg % 4 == 0 && c / 4 <= ROW_THREADS && ROW_THREADS % (c / 4) == 0 && al16(in);
    int nblocks;
    if (quads_form) {
        const int ppi = ROW_THREADS / (c / 4);
        nblocks = (hw + ppi - 1) / ppi;                         /* at least one step of the workgroup per block */
        if (nblocks > GN_MAX_BLOCKS) nblocks = GN_MAX_BLOCKS;
        const int per_block = (hw + nblocks - 1) / nblocks;
        nblocks = (hw + per_block - 1) / per_block;
        hipLaunchKernelGGL(k_gn_moments_quads, dim3(nblocks), dim3(ROW_THREADS), 0, st, part, in, hw, c, cg, per_block);
    } else {
        const size_t total = (size_t)hw * cg;
        nblocks = (int)((total + 4 * ROW_THREADS - 1) / (4 * ROW_THREADS));
        if (nblocks > GN_MAX_BLOCKS) nblocks = GN_MAX_BLOCKS;
        hipLaunchKernelGGL(k_gn_moments_any, dim3(groups, nblocks), dim3(ROW_THREADS), 0, st, part, in, hw, c, cg);
    }
    hipLaunchKernelGGL(k_gn_finish, dim3(groups), dim3(256), 0, st, stats, part, groups, nblocks, eps);
    const size_t n = (size_t)hw * c;
    if (al16(out) && al16(in) && al16(gamma) && al16(beta) && c % 4 == 0)
        hipLaunchKernelGGL(k_gn_normalize<4>, dim3(blocks_for(n, EW_THREADS * 4)), dim3(EW_THREADS), 0, st, out, in, stats, gamma, beta, c, cg, groups, do_silu, n);
    else
        hipLaunchKernelGGL(k_gn_normalize<1>, dim3(blocks_for(n, EW_THREADS)), dim3(EW_THREADS), 0, st, out, in, stats, gamma, beta, c, cg, groups, do_silu, n);
    return (int)hipGetLastError();
}

}  // extern "C"

/* ---- group norm for callers that cannot allocate -------------------------------------------
 * The same kernels with their scratch in a device array that is part of the library image, so the
 * call needs no hipMalloc: each GPU holds its own copy of the array, at its own address, until the
 * process ends. In host code the array's name is only a handle for hipGetSymbolAddress; kernels
 * get the address that call returned, kept per device. Calls on one GPU share the array: they must
 * not overlap (the library issues everything on one stream, which orders them). */
constexpr int GN_STATIC_MAX_GROUPS = IRIS_GN_MOST_GROUPS;
constexpr size_t GN_STATIC_FLOATS = SYNC_FLOATS + 3 * (size_t)GN_STATIC_MAX_GROUPS * GN_MAX_BLOCKS + 2 * (size_t)GN_STATIC_MAX_GROUPS;
static __device__ __align__(256) float scratch[GN_STATIC_FLOATS];          /* 1,052,288 B, zero when the library is loaded */

constexpr int GN_STATIC_MAX_DEVICES = 64;
static float *scratch_address[GN_STATIC_MAX_DEVICES];                        /* per device; null = not looked up yet */

extern "C" {

int iris_hip_group_norm_static_max_groups(void) { return GN_STATIC_MAX_GROUPS; }

/* Looks up the address of the current device's copy of the array (once per device). */
int iris_hip_group_norm_static_setup(void) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= GN_STATIC_MAX_DEVICES) return (int)hipErrorInvalidDevice;
    if (scratch_address[dev]) return 0;
    float *p = nullptr;
    e = hipGetSymbolAddress(reinterpret_cast<void **>(&p), HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (!p) return (int)hipErrorInvalidSymbol;
    scratch_address[dev] = p;
    return 0;
}

/* groups <= iris_hip_group_norm_static_max_groups(), checked by the caller too */
int iris_hip_group_norm_static(void *stream, float *out, const float *in, const float *gamma,
                               const float *beta, int hw, int c, int groups, float eps, int do_silu) {
    if (groups <= 0 || groups > GN_STATIC_MAX_GROUPS) return (int)hipErrorInvalidValue;
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= GN_STATIC_MAX_DEVICES) return (int)hipErrorInvalidDevice;
    if (!scratch_address[dev]) {                         /* first call on a device the set-up call did not see */
        const int rc = iris_hip_group_norm_static_setup();
        if (rc) return rc;
    }
    return iris_hip_group_norm(stream, scratch_address[dev], out, in, gamma, beta, hw, c, groups, eps, do_silu);
}

}  // extern "C"
