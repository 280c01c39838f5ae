/*
 * Linear layers whose 256-row tiles would leave the chip idle (reference iris_dev.h:48-53, iris_cuda.cu:456-505): the
 * short sequences of the text encoder, of the text rows of a double-stream block and of small pictures.
 *
 *   y[M, N] = x[M, K] @ W[N, K]^T      bf16 inputs, f32 accumulation, f32 or bf16 output
 *
 * With a few hundred rows a product has too few 256 x 256 tiles for 256 CUs (512 x 9728 -> 2560: 20), and each of its
 * workgroups then walks the whole of K alone. k_gemm_tiles takes smaller tiles and, where there are still too few, cuts
 * K into ranges that different workgroups multiply: each leaves f32 partial sums in a workspace and k_gemm_sum adds
 * them in order (no atomics: a call gives the same bits every time).
 *
 * A workgroup is WM x WN waves (eight, or four) of 16 NB rows x 16 NA columns, in KG groups: with KG = 2 both halves of the workgroup
 * own the same outputs and take one k-step of 32 each of every k tile of 64, and add their sums through the LDS at the
 * end. That keeps 64 x 64 outputs per wave, i.e. half an LDS read per product, on a tile of 128 x 128. W and x rows go
 * from memory straight into a ring of STAGES LDS stages (128 B rows, 16 B chunk c of row r in slot c ^ ((r >> 1) & 7),
 * which keeps the 128-bit reads off each other's banks, see k_gemm_dma); weights come from HBM here, so the ring is as
 * deep as the LDS allows. In front of the barrier of a k tile a wave waits for its own share of the next tile and for
 * its last operand reads of this one; behind it the stage is free and is requested again, STAGES tiles ahead.
 *
 * What bounds it is the fetch of the weights. A CU has at most the 32 KB of its vector cache in flight: rows from HBM
 * come at 50 GB/s a CU, rows from the L2 at 125 (direct loads by themselves, 32 to 64 workgroups on their own lines), and a
 * workgroup that only fetched its tiles and multiplied nothing took nine tenths of the whole kernel's time. The workgroups that
 * share W rows (one column of tiles) or x rows run in step, so each of them would wait for HBM for the same lines. Instead
 * they take the k tiles of a group of four in different orders (tile kt of the order is k tile kt ^ turn, turn = the tile's
 * row ^ its column, mod 4): a line is brought from HBM by one of them and found in the L2 by the others. Weights from HBM,
 * us, all in one order / turned: 512 x 2560 -> 6144 29.5 / 23.0, 512 x 3072 -> 9216 38.0 / 34.8, 512 x 9728 -> 2560 39.5 / 35.6,
 * 320 x 3072 -> 27648 59.1 / 55.5; with weights in the Infinity Cache 1 - 3 % slower, so not everywhere (iris_hip_gemm_turns).
 * The f32 sums of a row are then taken in an order that goes by its tile's place. Turns over eight tiles, or turned by pairs
 * and fours of tiles, gave the same or less; four waves that only fetch beside the eight that multiply changed nothing.
 * Then comes the LDS: a wave's 64 x 64 outputs read 8 KB of operands for 16 products. The tile of 160 x 224 runs on four waves of 80 x 112
 * (12 KB for 35 products; 512 registers to a wave) and fills 248 CUs with 320 x 3072 -> 27648 instead of 216: 58.0 us / 53.6. Tiles of
 * 160 x 256 on four waves are no faster than on eight, and their ends longer: 1000 x 3072 -> 9216 52.2 us on four / 52.1, -> 18432 105.6 / 103.8,
 * 11700 x 512 -> 1536 31.6 / 30.7, 1024 x 512 -> 1536 13.8 / 12.9.
 * Tiles of 128 x 256, 160 x 192 and 128 x 192 on four waves were as fast as on eight.
 * A tile of 128 x 96 is there for what its width fills the chip with: 512 x 2560 -> 6144 takes 256 workgroups instead of 192 of
 * 128 x 128, each of which fetches 224 rows instead of 256. Weights from HBM, us, without / with it: 512 x 2560 -> 6144 24.2 / 22.9,
 * 320 rows 25.3 / 22.6, 512 x 3072 -> 3072 22.4 / 20.2 (two ranges of K instead of three), 700 rows 26.0 / 23.2, 1000 x 4096 -> 2560
 * 32.2 / 30.2, 100 x 2560 -> 19456 33.0 / 30.7; no slower at any of the 60 sizes from 100 to 1000 rows where it is chosen.
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

constexpr int TK = 64;

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    f32x2 p = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(p, bf16x2));
}
__device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ uint32_t lds_address(const uint16_t *p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)p;
}

template <int NB, int WM, int NA, int WN, int KG, int STAGES>
struct Tile {
    static constexpr int TM = 16 * NB * WM, TN = 16 * NA * WN, WAVES = WM * WN * KG, THREADS = 64 * WAVES;
    static constexpr int STAGE = (TM + TN) * TK;                         /* elements: W rows, then x rows */
    static constexpr int PIECES = ((TM + TN) / 8 + WAVES - 1) / WAVES;   /* 8-row pieces a wave fetches per k tile */
    static constexpr int OUT_BYTES = WAVES * NB * 16 / KG * 256;         /* epilogue: rows of up to 64 f32 per wave */
    static constexpr int SUM_BYTES = KG == 2 ? WAVES * NB / 2 * NA * 1024 : 0;
    static constexpr int LDS = 2 * STAGES * STAGE > OUT_BYTES + SUM_BYTES ? 2 * STAGES * STAGE : OUT_BYTES + SUM_BYTES;
};

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"                          /* M0 in a clobber list */
template <typename OUT, int NB, int WM, int NA, int WN, int KG, int STAGES, bool THROUGH>
__global__ void __launch_bounds__(64 * WM * WN * KG, WM * WN * KG / 4)
k_gemm_tiles(OUT *__restrict__ y, const uint16_t *__restrict__ x, const uint16_t *__restrict__ W, int M, int N, int K,
             const float *__restrict__ bias, int tiles_m, int tiles_n, int splits, int total, int per_xcd, int turns) {
    using T = Tile<NB, WM, NA, WN, KG, STAGES>;
    constexpr int TM = T::TM, TN = T::TN, STAGE = T::STAGE, PIECES = T::PIECES;
    static_assert(T::LDS <= 160 * 1024 && NA <= 8 && (KG == 1 || (KG == 2 && NB % 2 == 0)), "");
    extern __shared__ __align__(16) uint16_t lds[];
    /* An XCD (own L2) takes a contiguous range of the work list: K ranges outermost, then bands of 8 tile rows, inside a
     * band m fastest: its 32 CUs share the W tiles and each other's x rows. */
    const int work = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (work >= total) return;
    constexpr int BAND = 8;
    const int per_split = tiles_m * tiles_n, split = work / per_split, in_split = work - split * per_split;
    const int band = in_split / (BAND * tiles_n), in_band = in_split - band * (BAND * tiles_n);
    const int band_rows = min(tiles_m - band * BAND, BAND);
    const int m0 = (band * BAND + in_band % band_rows) * TM, n0 = in_band / band_rows * TN;
    const int nk_all = K / TK, kt0 = (int)((long)nk_all * split / splits), nk = (int)((long)nk_all * (split + 1) / splits) - kt0;

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4;
    /* the order of this workgroup's k tiles, see above: tile kt of the order is k tile kt ^ turn inside whole groups of four */
    const int turn = (m0 / TM ^ n0 / TN) & turns, turned = nk & ~3;
    const int wm = wave % WM, wn = wave / WM % WN, kg = wave / (WM * WN);

    /* this wave's pieces of a stage: row 8 (PIECES wave + j) + lane / 8 of [W tile | x tile]; rows past the end of a matrix
     * repeat its last row (their outputs are never stored), pieces past the stage repeat its last piece */
    uint32_t off[PIECES];
    int piece[PIECES];
#pragma unroll
    for (int j = 0; j < PIECES; j++) {
        piece[j] = min(PIECES * wave + j, (TM + TN) / 8 - 1);
        const int r = 8 * piece[j] + (lane >> 3);
        const int row = r < TN ? min(n0 + r, N - 1) : min(m0 + r - TN, M - 1);
        off[j] = ((uint32_t)row * (uint32_t)K + 8u * ((lane & 7) ^ ((r >> 1) & 7))) * 2u;
    }
    auto request_one = [&](int j, int kt, uint16_t *stage) {
        const uint16_t *src = (piece[j] < TN / 8 ? W : x) + (size_t)(kt0 + (kt < turned ? kt ^ turn : kt)) * TK;
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     ::"s"(lds_address(stage + piece[j] * 8 * TK)), "v"(off[j]), "s"(src) : "memory", "m0");
    };
    /* waits for everything but the newest `tiles` requests and for the wave's LDS reads, then for the other waves */
    auto arrive = [&](int tiles) {
        if (tiles >= 3) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(3 * PIECES) : "memory");
        else if (tiles == 2) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * PIECES) : "memory");
        else if (tiles == 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(PIECES) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };

    f32x4 acc[NA][NB];
#pragma unroll
    for (int a = 0; a < NA; a++)
#pragma unroll
        for (int b = 0; b < NB; b++) acc[a][b] = f32x4{0, 0, 0, 0};
    u32x4 av[2][NA], bv[2][NB];
    int a_rd[2], b_rd[2];                                      /* [k-step], elements inside a stage */
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
        const int slot = 8 * ((4 * (KG == 2 ? kg : ks) + lg) ^ (li >> 1));
        a_rd[ks] = (16 * NA * wn + li) * TK + slot;
        b_rd[ks] = (TN + 16 * NB * wm + li) * TK + slot;
    }
    /* operand i of a k-step in the order the products use them: W block 0, the x blocks, the other W blocks */
    auto operand = [&](const uint16_t *stage, int set, int ks, int i) {
        if (i == 0 || i > NB) {
            const int a = i == 0 ? 0 : i - NB;
            av[set][a] = *reinterpret_cast<const u32x4 *>(&stage[a_rd[ks] + 16 * a * TK]);
        } else {
            bv[set][i - 1] = *reinterpret_cast<const u32x4 *>(&stage[b_rd[ks] + 16 * (i - 1) * TK]);
        }
    };
    /* A k-step's products with the memory instructions of later steps dealt out between them, at most one per gap: first
     * the operands of the next k-step (from `rd`, where `reads`), then, evenly, pieces [first, last) of a later k tile (`wanted`).
     * A wave issues in order, and the waves leave a barrier together: bunched in front of the products the same instructions
     * were not hidden by the other wave of the SIMD but added to it (128 x 256 tile: 1024 cycles of products, 1171 with
     * nothing else, 1477 with the operand reads, 1754 with the pieces too). */
    auto products = [&](int set, auto reads, const uint16_t *rd, int rd_ks, int first, int last, auto wanted, int kt, uint16_t *stage) {
        constexpr int GAPS = NA * NB, READS = NA + NB;
#pragma unroll
        for (int g = 0; g < GAPS; g++) {
            acc[g / NB][g % NB] = mfma(av[set][g / NB], bv[set][g % NB], acc[g / NB][g % NB]);
            if (decltype(reads)::value && g < READS) operand(rd, set ^ 1, rd_ks, g);
            const int gap = g - READS, span = GAPS - READS, count = last - first, j = gap * count / span;
            if (gap >= 0 && count && (gap == 0 || (gap - 1) * count / span != j))
                if (wanted) request_one(first + j, kt, stage);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    uint16_t *const ring_end = lds + STAGES * STAGE;
    for (int t = 0; t < STAGES && t < nk; t++)
#pragma unroll
        for (int j = 0; j < PIECES; j++) request_one(j, t, lds + t * STAGE);
    arrive(min(STAGES, nk) - 1);
#pragma unroll
    for (int i = 0; i < NA + NB; i++) operand(lds, 0, 0, i);
    uint16_t *prev = lds, *cur = lds, *nxt = lds + STAGE;
    auto advance = [&]() { prev = cur; cur = nxt; nxt = nxt + STAGE == ring_end ? lds : nxt + STAGE; };
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    int t = 0;
    if constexpr (KG == 1) {
        /* half of a tile's pieces behind the second half of the products of the tile whose stage it takes, half behind
         * the first half of the next tile's */
        auto tile = [&](auto first_half, auto second_half) {
            products(0, yes, cur, 1, PIECES / 2, PIECES, first_half, t - 1 + STAGES, prev);
            arrive(min(STAGES - 2, nk - 2 - t));
            products(1, yes, nxt, 0, 0, PIECES / 2, second_half, t + STAGES, cur);
            advance();
        };
        if (nk > 1) { tile(no, nk > STAGES); t++; }
        for (; t + STAGES < nk; t++) tile(yes, yes);
        for (; t + 1 < nk; t++) tile(t - 1 + STAGES < nk, no);
        products(0, yes, cur, 1, 0, 0, no, 0, cur);
        products(1, no, cur, 0, 0, 0, no, 0, cur);
    } else {
        auto tile = [&](int set, auto wanted) {
            arrive(min(STAGES - 2, nk - 2 - t));
            products(set, yes, nxt, 0, 0, PIECES, wanted, t + STAGES, cur);
            advance();
            t++;
        };
        while (t + 1 + STAGES < nk) {
            tile(0, yes);
            tile(1, yes);
        }
        while (t + 2 < nk) {
            tile(0, t + STAGES < nk);
            tile(1, t + STAGES < nk);
        }
        if (t + 1 < nk) {
            tile(0, t + STAGES < nk);
            products(1, no, cur, 0, 0, 0, no, 0, cur);
        } else {
            products(0, no, cur, 0, 0, 0, no, 0, cur);
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");          /* the ring is free */

    /* acc[a][b][r] = y[m0 + 16 (NB wm + b) + li][n0 + 16 (NA wn + a) + 4 lg + r]. With two k groups each keeps half of the
     * row blocks: it hands the other half to its partner and adds what it gets, group 0's sum first. */
    constexpr int NBS = NB / KG;                               /* row blocks this wave stores, from block b0 */
    const int b0 = kg * NBS;
    if constexpr (KG == 2) {
        f32x4 *sum = reinterpret_cast<f32x4 *>(reinterpret_cast<char *>(lds) + T::OUT_BYTES);
        f32x4 *mine = sum + (size_t)wave * NBS * NA * 64, *theirs = sum + (size_t)(wave ^ (WM * WN)) * NBS * NA * 64;
        static_assert((WM * WN & (WM * WN - 1)) == 0, "the partner is one bit away");
#pragma unroll
        for (int b = 0; b < NBS; b++)
#pragma unroll
            for (int a = 0; a < NA; a++) mine[(b * NA + a) * 64 + lane] = kg ? acc[a][b] : acc[a][NBS + b];
        __syncthreads();
#pragma unroll
        for (int b = 0; b < NBS; b++)
#pragma unroll
            for (int a = 0; a < NA; a++) {
                const f32x4 v = theirs[(b * NA + a) * 64 + lane];
                acc[a][b] = kg ? v + acc[a][NBS + b] : acc[a][b] + v;
            }
    }
    /* through the LDS (a region per wave, no barrier) so that a store instruction covers whole row segments */
    OUT *dst = y + (size_t)split * M * N;
    const int mw = m0 + 16 * (NB * wm + b0), nw = n0 + 16 * NA * wn;
    uint16_t *mine = lds + wave * (NBS * 16 * 128);
    /* up to 64 columns at a time */
#pragma unroll
    for (int c0 = 0; c0 < NA; c0 += 4) {
        const int na = min(NA - c0, 4), nc = nw + 16 * c0;
        if constexpr (sizeof(OUT) == 4) {
            float *buf = reinterpret_cast<float *>(mine);      /* 16 B chunk c of row r in slot c ^ (r % 16) */
#pragma unroll
            for (int b = 0; b < NBS; b++)
#pragma unroll
                for (int a = 0; a < na; a++) *reinterpret_cast<f32x4 *>(&buf[(16 * b + li) * 64 + 4 * ((4 * a + lg) ^ li)]) = acc[c0 + a][b];
#pragma unroll
            for (int it = 0; it < 4 * NBS; it++) {
                const int row = 4 * it + (lane >> 4), c = lane & 15, m = mw + row, n = nc + 4 * c;
                f32x4 v = *reinterpret_cast<const f32x4 *>(&buf[row * 64 + 4 * (c ^ (row & 15))]);
                if (c < 4 * na && m < M && n < N) {
                    if (bias) v += *reinterpret_cast<const f32x4 *>(bias + n);
                    if constexpr (THROUGH) store_through(dst + (size_t)m * N + n, v);
                    else *reinterpret_cast<f32x4 *>(dst + (size_t)m * N + n) = v;
                }
            }
        } else {
            uint16_t *buf = mine;                              /* chunk c of row r in slot c ^ (r % 8) */
#pragma unroll
            for (int b = 0; b < NBS; b++)
#pragma unroll
                for (int a = 0; a < na; a++) {
                    const int chunk = 2 * a + (lg >> 1);
                    *reinterpret_cast<uint2 *>(&buf[(16 * b + li) * 64 + 8 * (chunk ^ (li & 7)) + 4 * (lg & 1)]) =
                        make_uint2(pack_bf16(acc[c0 + a][b][0], acc[c0 + a][b][1]), pack_bf16(acc[c0 + a][b][2], acc[c0 + a][b][3]));
                }
#pragma unroll
            for (int it = 0; it < 2 * NBS; it++) {
                const int row = 8 * it + (lane >> 3), c = lane & 7, m = mw + row, n = nc + 8 * c;
                const u32x4 v = *reinterpret_cast<const u32x4 *>(&buf[row * 64 + 8 * (c ^ (row & 7))]);
                if (c < 2 * na && m < M && n < N) *reinterpret_cast<u32x4 *>(dst + (size_t)m * N + n) = v;
            }
        }
    }
}
#pragma clang diagnostic pop

/* y[i] = part[0][i] + part[1][i] + ..., four values a thread (n a multiple of 8). AT_ONCE (at most `splits`) sums are requested
 * before the first is used: what bounds it is the launch and one trip to memory, and one range after the other was a trip each. With
 * the layer in front of it, us, eight values a thread and one after the other / now: 512 x 9728 -> 2560 (6 ranges) 36.5 / 36.0,
 * 512 x 9216 -> 3072 (4) 39.7 / 38.9, 700 x 12288 -> 3072 (3) 62.2 / 61.1, 1000 x 9728 -> 2560 (3) 56.4 / 54.9; 100 and 320 rows the same. */
constexpr int SUM_MOST = 8;
template <typename OUT, int AT_ONCE>
__global__ void __launch_bounds__(256)
k_gemm_sum(OUT *__restrict__ y, const float *__restrict__ part, size_t n, int splits) {
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= n) return;
    f32x4 v[AT_ONCE];
#pragma unroll
    for (int s = 0; s < AT_ONCE; s++) v[s] = *reinterpret_cast<const f32x4 *>(part + s * n + i);
#pragma unroll
    for (int s = 1; s < AT_ONCE; s++) v[0] += v[s];
#pragma unroll 4
    for (int s = AT_ONCE; s < splits; s++) v[0] += *reinterpret_cast<const f32x4 *>(part + s * n + i);
    if constexpr (sizeof(OUT) == 4) *reinterpret_cast<f32x4 *>(y + i) = v[0];
    else *reinterpret_cast<uint2 *>(y + i) = make_uint2(pack_bf16(v[0][0], v[0][1]), pack_bf16(v[0][2], v[0][3]));
}

template <typename OUT, int AT_ONCE = SUM_MOST>
int launch_sum(hipStream_t st, OUT *y, const float *part, size_t n, int splits) {
    if constexpr (AT_ONCE > 2)
        if (splits < AT_ONCE) return launch_sum<OUT, AT_ONCE - 1>(st, y, part, n, splits);
    hipLaunchKernelGGL((k_gemm_sum<OUT, AT_ONCE>), dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, st, y, part, n, splits);
    return (int)hipGetLastError();
}

/* The order of the k tiles, a mask as iris_hip_gemm_turns gives it. In a grid of more than 512 tiles of 256 x 256 a projection may be
 * issued as k_gemm_wide that normalises its own tiles (iris_hip_linear_qknorm_plan), whose bits are to be those of the plain
 * layer: all k tiles in one order there. It gives up 2627 x 3072 -> 18432 258 -> 249 us, 1600 x 2560 -> 19456 143 -> 135. */
static int turns(int M, int N, int K, int wgs) {
    return (long)((M + 255) / 256) * ((N + 255) / 256) > 512 ? 0 : iris_hip_gemm_turns(wgs, (size_t)N * K * 2);
}

/* THROUGH is a template's choice: with a test in front of every store of one kernel, plain ones took 0.5 - 2 % longer. us, one kernel / two / one that
 * only stores plainly: 96 x 2560 -> 6144 16.12 / 15.74 / 15.79, 150 x 12288 -> 3072 29.27 / 29.04 / 28.99, 900 x 12288 -> 3072 77.6 / 76.6 / 76.7. */
template <typename OUT, int NB, int WM, int NA, int WN, int KG, int STAGES, bool THROUGH = false>
int launch_tiles(hipStream_t st, OUT *y, const uint16_t *x, const uint16_t *W, int M, int N, int K, const float *bias, int splits, bool through) {
    if constexpr (sizeof(OUT) == 4 && !THROUGH)
        if (through) return launch_tiles<OUT, NB, WM, NA, WN, KG, STAGES, true>(st, y, x, W, M, N, K, bias, splits, true);
    using T = Tile<NB, WM, NA, WN, KG, STAGES>;
    static bool configured = false;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_gemm_tiles<OUT, NB, WM, NA, WN, KG, STAGES, THROUGH>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, T::LDS);
        if (e != hipSuccess) return (int)e;
        configured = true;
    }
    const int tiles_m = (M + T::TM - 1) / T::TM, tiles_n = (N + T::TN - 1) / T::TN, total = tiles_m * tiles_n * splits, per_xcd = (total + 7) / 8;
    hipLaunchKernelGGL((k_gemm_tiles<OUT, NB, WM, NA, WN, KG, STAGES, THROUGH>), dim3((unsigned)per_xcd * 8), dim3(T::THREADS), T::LDS, st, y, x, W, M, N, K,
                       bias, tiles_m, tiles_n, splits, total, per_xcd, turns(M, N, K, total));
    return (int)hipGetLastError();
}

/* The tiles, and what a workgroup's k tile of 64 costs in us. Measured on 80 - 2115 rows with weights from HBM: `step` in a
 * grid of one round, where the chip is not at its power limit, `step_two` in two. `step_more`, for longer ones, is what decides
 * between these tiles and k_gemm_wide, which is the faster one there unless its tiles fit badly; with the figures of two rounds
 * these tiles were taken for 12800 x 12288 -> 3072 (752 us on k_gemm_wide, 819 here), 9280 x 12288 -> 4096 (749 / 808),
 * 7176 x 16384 -> 4096 (734 / 804), 3680 x 4096 -> 36864 (862 / 900). A workgroup's first tiles and its epilogue take 3.5 us more.
 * Three digits where sizes are decided by them: 528 - 640 x 4096 -> 2560 24.4 us in four ranges of 160 x 192, 26.2 in five of 128 x 256.
 * `through`: see iris_hip_gemm_tiles_through. */
struct Shape { int tm, tn; float step, step_two, step_more; int through; };
constexpr Shape SHAPES[] = {{128, 128, 0.44f, 0.50f, 0.55f, 100}, {128, 192, 0.58f, 0.62f, 0.65f, 100}, {128, 256, 0.736f, 0.80f, 0.82f, 100},
                            {64, 256, 0.60f, 0.61f, 0.62f, 80},   {160, 192, 0.665f, 0.72f, 0.74f, 64}, {160, 256, 0.90f, 0.93f, 0.94f, 64},
                            {160, 224, 0.836f, 0.87f, 0.89f, 64}, {128, 96, 0.39f, 0.45f, 0.50f, 64}};
constexpr int NSHAPES = sizeof(SHAPES) / sizeof(SHAPES[0]);

template <typename OUT>
int launch_shape(hipStream_t st, int shape, OUT *y, const uint16_t *x, const uint16_t *W, int M, int N, int K, const float *bias, int splits,
                 bool through = false) {
    switch (shape) {
    case 0: return launch_tiles<OUT, 4, 2, 4, 2, 2, 4>(st, y, x, W, M, N, K, bias, splits, through);
    case 1: return launch_tiles<OUT, 4, 2, 3, 4, 1, 4>(st, y, x, W, M, N, K, bias, splits, through);
    case 2: return launch_tiles<OUT, 4, 2, 4, 4, 1, 3>(st, y, x, W, M, N, K, bias, splits, through);
    case 3: return launch_tiles<OUT, 4, 1, 4, 4, 2, 4>(st, y, x, W, M, N, K, bias, splits, through);
    case 4: return launch_tiles<OUT, 5, 2, 3, 4, 1, 3>(st, y, x, W, M, N, K, bias, splits, through);
    case 5: return launch_tiles<OUT, 5, 2, 4, 4, 1, 3>(st, y, x, W, M, N, K, bias, splits, through);
    case 6: return launch_tiles<OUT, 5, 2, 7, 2, 1, 3>(st, y, x, W, M, N, K, bias, splits, through);
    case 7: return launch_tiles<OUT, 4, 2, 3, 2, 2, 4>(st, y, x, W, M, N, K, bias, splits, through);
    default: return (int)hipErrorInvalidValue;
    }
}

}  // namespace

extern "C" {

/* 3: the workgroups of a product take the k tiles of a group of four in different orders (the mask of the turn), 0: all in one.
 * The first brings new lines from HBM once; on lines that are already on the chip it is only a cost. So the weights have to be
 * larger than an XCD's L2 (4 MB) even in a grid of one round, larger than 14 MB in a longer one, whose later rounds find smaller
 * ones on the chip. Weights from HBM, us, one order / turned: 512 x 1536 -> 4096
 * (12 MB, one round) 16.3 / 13.9, 1500 x 2560 -> 2560 29.0 / 24.5, 512 x 1024 -> 4096 (8 MB) 11.7 / 10.7; more rounds:
 * 3000 x 512 -> 8192 (8 MB) 29.5 / 30.8, 9000 x 768 -> 6272 81.3 / 83.2, 14650 x 512 -> 6912 109.1 / 111.6, 3179 x 512 -> 15488 (15 MB)
 * 61.7 / 57.2, 2692 x 1024 -> 18944 106.8 / 103.4; 2 MB, 14391 x 512 -> 1536 31.6 / 32.5, and the VAE's attention block on weights
 * of 1.5 MB 576 / 582. The other way: 2115 x 512 -> 8192 27.3 / 25.2. */
int iris_hip_gemm_turns(long wgs, size_t weight_bytes) { return weight_bytes > (size_t)(wgs <= 256 ? 4 : 14) << 20 ? 3 : 0; }

/* 1: this tile adds the products of an output one k-step after the other, as k_gemm_wide does in one order (KG = 1, K whole) */
int iris_hip_gemm_tiles_in_order(int shape, int splits, int M, int N, int K) {
    constexpr bool two_groups[NSHAPES] = {true, false, false, true, false, false, false, true};
    const long wgs = (long)((M + SHAPES[shape].tm - 1) / SHAPES[shape].tm) * ((N + SHAPES[shape].tn - 1) / SHAPES[shape].tn);
    return splits == 1 && !two_groups[shape] && turns(M, N, K, (int)(wgs < 1 << 30 ? wgs : 1 << 30)) == 0;
}

/* 1: the partial sums of a product in ranges of K leave the L2s as they are stored (write_through.h) and not in front of the sum: those of
 * up to 20 MB, with weights of up to `through` MB. Larger weights, of which a single row of tiles takes a new line with every load, are
 * slowed down by the stores beside them, from different sizes on with each tile. us, all plain / all through, weights from HBM, up to the bound:
 * 64 x 9728 -> 2560 (48 MB) 19.5 / 18.1, 128 x 9216 -> 3072 (54) 21.3 / 20.4, 64 x 12288 -> 3072 (72) 23.5 / 22.8, 90 rows 26.6 / 25.7, 72 x 3072 -> 15360
 * (90) 28.4 / 27.3, 100 x 4096 -> 12288 (96) 33.8 / 32.6, 128 x 12288 -> 4096 30.2 / 28.9; beyond it 123 x 12288 -> 3072 (tiles of 128 x 96) 25.1 / 25.7, 64 x
 * 3072 -> 15360 (64 x 256) 26.8 / 27.3, 64 x 2560 -> 19456 (95 MB) 28.0 / 28.7, 129 rows (160 x 192) 33.7 / 35.0, 64 x 3072 -> 18432 (108) 29.2 / 30.0, 128 x
 * 4096 -> 16384 (128) 43.5 / 44.1, 128 x 5120 -> 13824 (135) 39.8 / 41.0, 100 x 13824 -> 5120 37.8 / 38.6. 159 products of 16 to 768 rows up to both bounds
 * are 0.9 to 8 % faster, half of them by 4 % or more; of 72 up to 20 MB beyond the other, half are slower, by up to 4 %. */
int iris_hip_gemm_tiles_through(int shape, int splits, int M, int N, int K) {
    return splits > 1 && (size_t)splits * M * N * 4 <= (size_t)20 << 20 && (size_t)N * K * 2 <= (size_t)SHAPES[shape].through << 20;
}

/* The cheapest tile and number of K ranges for a product, and its estimated time in us; negative where these kernels do
 * not take it: they want rows of 16-byte chunks (N % 8), whole k tiles and enough of them to fill the ring, and 32-bit
 * byte offsets. Partial sums take splits * M * N floats of the workspace. Host arithmetic only. */
float iris_hip_gemm_tiles_plan(int M, int N, int K, int out_size, size_t part_bytes, int *shape, int *splits) {
    constexpr int MIN_TILES = 6;                               /* k tiles of a range */
    if (M <= 0 || N < 128 || N % 8 || K % TK || K < 8 * TK || ((size_t)M * K * 2) >> 32 || ((size_t)N * K * 2) >> 32) return -1.0f;
    const int nk = K / TK;
    float best = -1.0f;
    for (int i = 0; i < NSHAPES; i++) {
        const long tiles = (long)((M + SHAPES[i].tm - 1) / SHAPES[i].tm) * ((N + SHAPES[i].tn - 1) / SHAPES[i].tn);
        for (int s = 1; s == 1 || (s * MIN_TILES <= nk && (size_t)s * M * N * 4 <= part_bytes && tiles * s <= 512); s++) {
            const long wgs = tiles * s, rounds = (wgs + 255) / 256;
            /* Rows of a multiple of 32 KB cut into ranges of a multiple of 4 KB: the lines that a single row of tiles fetches at a time
             * lie as far apart, and come slower. 112 x 16384 -> 4096 in eight ranges of 128 x 128 41.7 us, 16448 -> 4096 36.6; in
             * sixteen of 128 x 256 36.9. */
            const float far_apart = M <= SHAPES[i].tm && K % 16384 == 0 && ((nk + s - 1) / s) % 32 == 0 ? 1.3f : 1.0f;
            const float step = rounds > 2 ? SHAPES[i].step_more : rounds > 1 ? SHAPES[i].step_two : SHAPES[i].step;
            /* the sum: a launch, and its reads at 5 TB/s */
            const float sum = s > 1 ? 3.0f + ((float)s * 4.0f + (float)out_size) * (float)M * (float)N / 5e6f : 0.0f;
            const float cost = 4.0f + (float)rounds * ((float)((nk + s - 1) / s) * step * far_apart + 3.5f) + sum;
            if (best < 0.0f || cost < best) { best = cost; *shape = i; *splits = s; }
        }
    }
    return best;
}

/* part: splits * M * N floats, 16-byte aligned, when splits > 1. x, W, y, bias 16-byte aligned; bias (or null) [N], with f32
 * outputs and one range only. */
int iris_hip_gemm_tiles(void *stream, void *y, int out_size, const uint16_t *x, const uint16_t *W, int M, int N, int K, const float *bias, int shape,
                        int splits, float *part) {
    hipStream_t st = (hipStream_t)stream;
    if (splits == 1)
        return out_size == 2 ? launch_shape<uint16_t>(st, shape, (uint16_t *)y, x, W, M, N, K, nullptr, 1)
                             : launch_shape<float>(st, shape, (float *)y, x, W, M, N, K, bias, 1);
    int e = launch_shape<float>(st, shape, part, x, W, M, N, K, nullptr, splits, iris_hip_gemm_tiles_through(shape, splits, M, N, K) != 0);
    if (e) return e;
    const size_t n = (size_t)M * N;
    return out_size == 2 ? launch_sum(st, (uint16_t *)y, part, n, splits) : launch_sum(st, (float *)y, part, n, splits);
}

}  // extern "C"
