// Generic MLX-affine INT4 GEMV over weights in the reference's row-major layout (W uint8 [m][n/2],
// bf16 scale/bias per 64): y[r] = W x[r] for 1..16 input rows against one read of W.
//
// Replaces dequant_int4_gemv_simd / dequant_int4_gemv_rows (Metal/Quant/dequant_int4.metal:78-357) and
// the LM-head row GEMV (Metal/Sampling/logit.metal:614-667).
//
// A wave owns kRowsPerWave consecutive weight rows. Lane l owns the 16-byte chunks l, l + 64, ... of
// every row (32 nibbles = half a group each), so one load instruction covers 1 KiB of a row and the
// input values a lane needs are the same for all of its rows: they are loaded once per chunk round,
// paired as (x[m], x[m+4]) to line up with ((w >> 4m) & 0x000F000F), and reused for every weight row.
// Per chunk: acc = sum (128 + q) x by v_dot2_f32_bf16, then s * acc + (b - 128 s) * sum x, the factored
// form of dequant_int4.metal:104-139. Rows are reduced across the wave by a xor-butterfly.
// That kernel serves rows longer than a wave's K-slice holds; up to FFMOE_MATRIX_MAX_N the sums run on the matrix unit
// (gemv_int4_mfma_kernel below).
// Each input row accumulates independently of the others, so row r of a multi-row call equals the
// single-row call bit for bit (the property DequantInt4SmallBatchTests.swift:74-78 asserts).
#include "common.hpp"
#include "kernels.hpp"
#include "stream.hpp"

namespace ffmoe {
namespace {

constexpr int kRowsPerWave = 8;
constexpr int kRowTile = 4;   // input rows held in registers per pass

template <bool F16>
__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c) {
    if constexpr (F16) return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, a), __builtin_bit_cast(f16x2, b), c, false);
    else return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b), c, false);
}

template <bool ALIGNED>
__device__ __forceinline__ uint4 load_chunk(const uint8_t *p) {
    if (ALIGNED) return *reinterpret_cast<const uint4 *>(p);
    const uint16_t *h = reinterpret_cast<const uint16_t *>(p);   // 2-byte alignment is guaranteed
    uint4 r;
    r.x = (uint32_t)h[0] | ((uint32_t)h[1] << 16);
    r.y = (uint32_t)h[2] | ((uint32_t)h[3] << 16);
    r.z = (uint32_t)h[4] | ((uint32_t)h[5] << 16);
    r.w = (uint32_t)h[6] | ((uint32_t)h[7] << 16);
    return r;
}

// eight consecutive bf16 inputs as four dwords
template <bool X_ALIGNED>
__device__ __forceinline__ uint4 load_x8(const uint16_t *src) {
    if (X_ALIGNED) return *reinterpret_cast<const uint4 *>(src);
    uint4 r;
    r.x = (uint32_t)src[0] | ((uint32_t)src[1] << 16);
    r.y = (uint32_t)src[2] | ((uint32_t)src[3] << 16);
    r.z = (uint32_t)src[4] | ((uint32_t)src[5] << 16);
    r.w = (uint32_t)src[6] | ((uint32_t)src[7] << 16);
    return r;
}

// F16: inputs and 16-bit outputs are FP16 (a context in FP16 mode); the offset form is then 1024 + q
template <bool ALIGNED, bool X_ALIGNED, bool Y_F32, bool F16>
__global__ __launch_bounds__(256) void gemv_int4_kernel(const uint8_t *__restrict__ w, const uint16_t *__restrict__ scales,
                                                        const uint16_t *__restrict__ biases,
                                                        const uint16_t *__restrict__ x, void *__restrict__ y_,
                                                        uint32_t m, uint32_t n, uint32_t rows, uint32_t x_stride,
                                                        uint32_t y_stride, const uint32_t *__restrict__ ids) {
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t m0 = (blockIdx.x * 4 + wave) * kRowsPerWave;
    if (m0 >= m) return;
    // output o is weight row o, or row ids[o] of the table when a list is given (encodeRowsListed)
    uint32_t wrow[kRowsPerWave];
#pragma unroll
    for (int mi = 0; mi < kRowsPerWave; ++mi) {
        const uint32_t o = min(m0 + mi, m - 1);
        wrow[mi] = ids ? ids[o] : o;
    }
    const uint32_t row_bytes = n / 2, n_groups = n / kGroup, chunks = n / 32;
    const uint32_t rounds = (chunks + 63) / 64;

    for (uint32_t r0 = 0; r0 < rows; r0 += kRowTile) {
        float acc[kRowsPerWave][kRowTile];
#pragma unroll
        for (int mi = 0; mi < kRowsPerWave; ++mi)
#pragma unroll
            for (int r = 0; r < kRowTile; ++r) acc[mi][r] = 0.0f;

        for (uint32_t j = 0; j < rounds; ++j) {
            const uint32_t c = lane + 64 * j;
            if (c >= chunks) continue;
            // input values of this chunk, paired (x[e], x[e+4]) per run of eight, and their sum
            uint32_t xp[kRowTile][16];
            float sx[kRowTile];
#pragma unroll
            for (int r = 0; r < kRowTile; ++r) {
                const uint32_t row = min(r0 + r, rows - 1);
                const uint16_t *src = x + (size_t)row * x_stride + (size_t)c * 32;
                float sum = 0.0f;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint4 dv = load_x8<X_ALIGNED>(src + q * 8);
                    const uint32_t d[4] = {dv.x, dv.y, dv.z, dv.w};
                    xp[r][q * 4 + 0] = (d[0] & 0xFFFFu) | (d[2] << 16);
                    xp[r][q * 4 + 1] = (d[0] >> 16) | (d[2] & 0xFFFF0000u);
                    xp[r][q * 4 + 2] = (d[1] & 0xFFFFu) | (d[3] << 16);
                    xp[r][q * 4 + 3] = (d[1] >> 16) | (d[3] & 0xFFFF0000u);
#pragma unroll
                    for (int i = 0; i < 4; ++i) { sum += Act<F16>::lo(d[i]); sum += Act<F16>::hi(d[i]); }
                }
                sx[r] = sum;
            }
            uint4 wv[kRowsPerWave];
            uint32_t sb[kRowsPerWave];
#pragma unroll
            for (int mi = 0; mi < kRowsPerWave; ++mi) {
                const uint32_t row = wrow[mi];
                wv[mi] = load_chunk<ALIGNED>(w + (size_t)row * row_bytes + (size_t)c * 16);
                const size_t gi = (size_t)row * n_groups + (c >> 1);
                sb[mi] = (uint32_t)scales[gi] | ((uint32_t)biases[gi] << 16);
            }
#pragma unroll
            for (int mi = 0; mi < kRowsPerWave; ++mi) {
                uint32_t q[16];
                const uint32_t ww[4] = {wv[mi].x, wv[mi].y, wv[mi].z, wv[mi].w};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
#pragma unroll
                    for (int p = 0; p < 4; ++p) q[i * 4 + p] = ((ww[i] >> (4 * p)) & 0x000F000Fu) | Act<F16>::kOffsetBits;
                }
                const float s = bf16lo_to_f32(sb[mi]), b = bf16hi_to_f32(sb[mi]);
                const float tb = __builtin_fmaf(-Act<F16>::kOffset, s, b);
#pragma unroll
                for (int r = 0; r < kRowTile; ++r) {
                    float dsum = 0.0f;
#pragma unroll
                    for (int p = 0; p < 16; ++p) dsum = dot2<F16>(q[p], xp[r][p], dsum);
                    acc[mi][r] = __builtin_fmaf(s, dsum, acc[mi][r]);
                    acc[mi][r] = __builtin_fmaf(tb, sx[r], acc[mi][r]);
                }
            }
        }
#pragma unroll
        for (int mi = 0; mi < kRowsPerWave; ++mi) {
#pragma unroll
            for (int r = 0; r < kRowTile; ++r) {
                const float v = wave_butterfly_sum_shuffle(acc[mi][r]);
                if (lane == 0 && m0 + mi < m && r0 + r < rows) {
                    const size_t o = (size_t)(r0 + r) * y_stride + m0 + mi;
                    if (Y_F32) reinterpret_cast<float *>(y_)[o] = v;
                    else reinterpret_cast<uint16_t *>(y_)[o] = Act<F16>::round(v);
                }
            }
        }
    }
}

// The same product on the matrix unit, for n <= kListedParts * kListedRing * 64. A block takes 16 weight rows at a time, its eight waves split
// K; a group's product is v_mfma_f32_16x16x32 of the (up to 16) input rows with the nibbles as 16 + q (bf16) or as
// subnormals (FP16: common.hpp), then s * acc + (b - 16 s) * sum x, as in the expert kernels (stream.hpp) but on the reference's row-major bytes: four
// neighbouring lanes load the 32 bytes of a row's group (16 segments per request instead of 64) and ds_bpermute hands
// each operand lane (row i, quarter q) its eight bytes, the values k = 16 q .. 16 q + 15 of the group. Nibble p of such a
// dword is element p, so ((w >> 4 m) & 0x000F000F) pairs elements m and m + 4, and the input operand is paired the same way.
// FEW (up to four input rows): input row t is operand row 4 t, so that one of a lane's four sums is all there is to keep up, and
// each operand lane loads its own bytes - the lanes of a row ask for the same ones, nothing is turned through LDS.
// Bound: latency - row id, weights, products and the merge are one chain per 16 rows, and a hot list of a few thousand
// rows is one such chain per compute unit. So eight waves take six groups each: with four, eleven each, a chain was twice as long and
// a block's registers left two waves per SIMD. Listed rows x 2,816, us with four waves | eight: 512 rows, 1 input row 6.4 | 4.8;
// 4,099 rows, 1 input row 7.1 | 5.7, 16 input rows 7.4 | 6.2 (all shorter still, below; the vector unit's dot products: 50.8); 32,768 rows 17.7 | 16.8, 19.0 | 17.5.
// EARLY (but for lists of more than a block per 16 rows with more than four input rows): the input rows are asked for while the ids are on their way, and
// the scales and all six groups of weights in one burst: of up to four input rows as soon as the ids are there, of more once the input rows are
// there too and turned, in front of their sums. (16 segments per request, they would stand behind the weights of the block's earlier waves in the unit's
// cache, which keeps its order: 16 input rows, weights that no cache holds, us with the turn behind the burst | in front: 512 listed rows 4.45 | 4.28, 1,408 4.76 | 4.57,
// 4,096 5.09 | 4.79, 4,099 6.50 | 6.32, 8,192 7.70 | 7.25. With up to four it is 4.36 behind and 4.42 in front at 1,408.) Left alone the compiler asks for
// the weights behind the sums and, ONE, two or three groups at a time where it uses them, each a round trip to memory. Us of the call so | now,
// of lists that repeat and of rows that no cache holds: 512 rows, 4 input rows 4.24 | 4.20 and 4.65 | 4.27, 16 input rows 4.40 | 4.22 and 4.86 | 4.28;
// 1,408 rows 4.25 | 4.15 and 5.22 | 4.28, 4.42 | 4.22 and 5.26 | 4.57; 4,096 rows 4.17 | 4.15 and 5.47 | 4.55, 4.63 | 4.25 and 5.42 | 4.79. Where units have two
// blocks, 4,099 rows (one unit) 4.68 | 4.93 and 5.83 | 5.48, 5.66 | 5.65 and 6.16 | 6.33, 5,120 rows 5.09 | 5.32 and 6.77 | 6.23, 6.08 | 6.07 and 6.95 | 6.95, 8,192
// rows 5.43 | 5.38 and 7.05 | 6.53, 6.29 | 6.13 and 8.08 | 7.25. More than a block per 16 rows: 16,384 rows, 4 input rows 9.80 | 9.43 and 11.19 | 11.06, 32,768 rows 14.80 | 14.95 and
// 17.67 | 17.17; with 16 input rows the weights behind the sums are the faster: 9.6 and 12.0, in front of them 10.1 and 12.6.
// Error of a logit against 64 bits (2-norm): 1.7e-7 in bf16 and 4.9e-6 in FP16, where the dot products have
// 8.6e-7 and 1.6e-5, and 128 + q / 1024 + q on the matrix unit 1.0e-6 and 1.4e-5.
constexpr int kListedParts = 8, kListedRing = 6;
static_assert(kListedParts * kListedRing >= kKSplit * kRing, "every width up to FFMOE_MATRIX_MAX_N");
// ONE: the launch has a block for every 16 rows, none of which takes others: it asks for no further weights, whose requests (the same rows
// again) a block would have to wait for before it can end. Us of the call with the requests (and the weights behind the sums) | so, of lists that repeat and of
// rows that no cache holds: 1,408 rows, 4 input rows 4.32 | 4.15 and 5.18 | 4.28, 16 input rows 4.75 | 4.22 and 5.49 | 4.57; 4,099 rows 5.68 | 4.93 and 6.25 | 5.48,
// 5.91 | 5.65 and 6.29 | 6.33; 8,192 rows 7.10 | 5.38 and 8.20 | 6.53, 7.09 | 6.13 and 8.95 | 7.25. Beyond, two blocks per compute unit go on to others.
template <bool ALIGNED, bool X_ALIGNED, bool Y_F32, bool F16, bool FEW, bool ONE>
__global__ __launch_bounds__(64 * kListedParts, 4) void gemv_int4_mfma_kernel(const uint8_t *__restrict__ w, const uint16_t *__restrict__ scales,
                                                                              const uint16_t *__restrict__ biases, const uint16_t *__restrict__ x,
                                                                              void *__restrict__ y_, uint32_t m, uint32_t n_groups, uint32_t rows,
                                                                              uint32_t x_stride, uint32_t y_stride, const uint32_t *__restrict__ ids) {
    constexpr int kSums = FEW ? 1 : 4;
    constexpr bool EARLY = FEW || ONE;                              // (without a branch from here to the first products)
    __shared__ float s_red[ONE ? 1 : 2][kListedParts][kSums][64];
    const uint32_t lane = threadIdx.x & 63, ks = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t j = lane & 15, jq = lane >> 4;                  // operand layout: row j, quarter jq
    const uint32_t lrow = lane >> 2, lq = lane & 3;                // load layout: row lrow, quarter lq
    const uint32_t n_blocks = (m + kTileRows - 1) / kTileRows;
    const uint32_t g0 = ks * n_groups / kListedParts, ng = (ks + 1) * n_groups / kListedParts - g0;
    const uint32_t g_last = ng ? g0 + ng - 1 : min(g0, n_groups - 1);
    const size_t row_bytes = (size_t)n_groups * (kGroup / 2);
    auto id_of = [&](uint32_t rb) {
        const uint32_t o = min(rb * kTileRows + lrow, m - 1);
        return ids ? ids[o] : o;
    };
    // As they come from memory: what a word is put together from stays apart until it is used, so that no load waits for one before it.
    struct Words { uint32_t part[ALIGNED ? 2 : 4]; };               // ALIGNED: two words, else (2-byte alignment is guaranteed) their halves
    Words wt[kListedRing];
    uint2 first_sb[2];                                              // scale and bias of groups g0 + 2 lq + 0 .. 1 of row lrow
    auto load_w = [&](uint32_t row, int u) {
        const uint8_t *p = w + row * row_bytes + (size_t)min(g0 + u, g_last) * (kGroup / 2) + 8 * lq;
        Words r;
        if constexpr (ALIGNED) {
            const uint2 v = *reinterpret_cast<const uint2 *>(p);
            r.part[0] = v.x, r.part[1] = v.y;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) r.part[i] = reinterpret_cast<const uint16_t *>(p)[i];
        }
        return r;
    };
    auto word = [](const Words &r, int i) { return ALIGNED ? r.part[i] : r.part[2 * i % 4] | (r.part[(2 * i + 1) % 4] << 16); };
    auto load_s = [&](uint32_t row, int v) {
        const size_t at = (size_t)row * n_groups + min(g0 + 2 * lq + v, g_last);
        return make_uint2(scales[at], biases[at]);
    };
    auto pair = [](const uint2 &v) { return v.x | (v.y << 16); };
    uint32_t rb = blockIdx.x;
    if (EARLY && rb >= n_blocks) return;                            // (the grid has at most n_blocks blocks: the loop's first turn needs no test)
    uint32_t row = id_of(rb), next_id = ONE ? 0u : id_of(min(rb + gridDim.x, n_blocks - 1));
    // the input rows of this wave's K-slice
    uint4 x0[kListedRing], x1[kListedRing];
    {
        const uint32_t my = FEW ? j >> 2 : lrow, quarter = FEW ? jq : lq;
        const uint16_t *xrow = x + (size_t)min(my, rows - 1) * x_stride + 16 * quarter;
#pragma unroll
        for (int u = 0; u < kListedRing; ++u) {
            const uint16_t *p = xrow + min(g0 + u, g_last) * kGroup;
            const bool ask = EARLY || (uint32_t)u < ng;             // (EARLY: past the share its last group again, whose products are left out below)
            x0[u] = ask ? load_x8<X_ALIGNED>(p) : uint4{0, 0, 0, 0};
            x1[u] = ask ? load_x8<X_ALIGNED>(p + 8) : uint4{0, 0, 0, 0};
        }
    }
    if constexpr (EARLY) __builtin_amdgcn_sched_barrier(0);
    if constexpr (!FEW) turn_token_rows(lane, x0, x1);              // ... in operand order
    if constexpr (!FEW && EARLY) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kListedRing; ++u) wt[u] = load_w(row, u);
#pragma unroll
    for (int v = 0; v < 2; ++v) first_sb[v] = load_s(row, v);
    if constexpr (EARLY) __builtin_amdgcn_sched_barrier(0);
    // ... paired like the nibbles, and their sum per group
    f32x4 sx[kListedRing];
    {
        auto paired = [](const uint4 &d) {
            return uint4{(d.x & 0xFFFFu) | (d.z << 16), (d.x >> 16) | (d.z & 0xFFFF0000u),
                         (d.y & 0xFFFFu) | (d.w << 16), (d.y >> 16) | (d.w & 0xFFFF0000u)};
        };
#pragma unroll
        for (int u = 0; u < kListedRing; ++u) {
            x0[u] = paired(x0[u]);
            x1[u] = paired(x1[u]);
            sx[u] = group_input_sum<F16>(x0[u], x1[u]);
        }
    }
    if constexpr (EARLY) __builtin_amdgcn_sched_barrier(0);
    uint32_t sb[2] = {pair(first_sb[0]), pair(first_sb[1])};
    const int pull = (int)((4 * j + jq) * 4);
    const uint32_t my_row = FEW ? jq : 4 * jq + ks;                 // the input row this lane finishes (waves kSums and up: none)
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    for (int buf = 0; rb < n_blocks; rb += gridDim.x, buf ^= 1) {
        if constexpr (!ONE) {
            row = next_id;
            next_id = id_of(min(rb + 2 * gridDim.x, n_blocks - 1));
        }
        float tot[kSums];
#pragma unroll
        for (int r = 0; r < kSums; ++r) tot[r] = 0.0f;
#pragma unroll
        for (int u = 0; u < kListedRing; ++u) {
            uint2 t;
            t.x = (uint32_t)__builtin_amdgcn_ds_bpermute(pull, (int)word(wt[u], 0));
            t.y = (uint32_t)__builtin_amdgcn_ds_bpermute(pull, (int)word(wt[u], 1));
            uint32_t sc = (uint32_t)__builtin_amdgcn_ds_bpermute((int)((4 * j + u / 2) * 4), (int)sb[u % 2]);
            if (!EARLY && (uint32_t)u >= ng) sc = 0;
            if constexpr (!ONE) wt[u] = load_w(row, u);             // the next 16 rows (past the last: these again)
            f32x4 acc = Act<F16>::mfma(x0[u], unpack8_fine<F16>(t.x), zero);
            acc = Act<F16>::mfma(x1[u], unpack8_fine<F16>(t.y), acc);
            const float s = bf16lo_to_f32(sc), b = bf16hi_to_f32(sc), su = s * FineNibble<F16>::kUnit;
            const float tb = __builtin_fmaf(-FineNibble<F16>::kOffset, s, b);
#pragma unroll
            for (int r = 0; r < kSums; ++r) {
                const float sum = __builtin_fmaf(tb, sx[u][r], __builtin_fmaf(su, acc[r], tot[r]));
                tot[r] = !EARLY || (uint32_t)u < ng ? sum : tot[r];
            }
        }
        if constexpr (!ONE) {
#pragma unroll
            for (int v = 0; v < 2; ++v) sb[v] = pair(load_s(row, v));
        }
#pragma unroll
        for (int r = 0; r < kSums; ++r) s_red[buf][ks][r][lane] = tot[r];
        lds_barrier();
        if (ks >= (uint32_t)kSums) {
            if constexpr (ONE) return;
            continue;
        }
        float v = s_red[buf][0][ks][lane];
#pragma unroll
        for (int o = 1; o < kListedParts; ++o) v += s_red[buf][o][ks][lane];
        const uint32_t out = rb * kTileRows + j;
        if (my_row < rows && out < m) {
            const size_t at = (size_t)my_row * y_stride + out;
            if (Y_F32) reinterpret_cast<float *>(y_)[at] = v;
            else reinterpret_cast<uint16_t *>(y_)[at] = Act<F16>::round(v);
        }
        if constexpr (ONE) return;
    }
}

}  // namespace

hipError_t launch_gemv_int4(hipStream_t s, const uint8_t *w, const uint16_t *scales, const uint16_t *biases,
                            const uint16_t *x, void *y, uint32_t m, uint32_t n, uint32_t rows,
                            uint32_t x_stride, uint32_t y_stride, int y_f32, const uint32_t *ids, bool f16, uint32_t n_cus) {
    if (n <= FFMOE_MATRIX_MAX_N) {
        // every row count of such a width takes this form (the rows of a call equal single-row calls bit for bit)
        const uint32_t tiles = (m + kTileRows - 1) / kTileRows;
        const dim3 blocks(min(tiles, 2 * n_cus));
        const bool one = tiles <= 2 * n_cus;                 // a block for every 16 rows
        const bool wide_w = reinterpret_cast<uintptr_t>(w) % 8 == 0, wide_x = reinterpret_cast<uintptr_t>(x) % 16 == 0 && x_stride % 8 == 0;
        if (f16 && !wide_x) return hipErrorInvalidValue;     // FP16 rows come 16-byte aligned (checked at the boundary)
#define FFMOE_GEMVM(A, X, Y, H)                                                                                                     \
    hipLaunchKernelGGL((rows <= 4 ? (one ? gemv_int4_mfma_kernel<A, X, Y, H, true, true> : gemv_int4_mfma_kernel<A, X, Y, H, true, false>)     \
                                  : (one ? gemv_int4_mfma_kernel<A, X, Y, H, false, true> : gemv_int4_mfma_kernel<A, X, Y, H, false, false>)), blocks, \
                       dim3(64 * kListedParts), 0, s, w, scales, biases, x, y, m, n / kGroup, rows, x_stride, y_stride, ids)
#define FFMOE_GEMVM_X(A, Y)                                                                             \
    do {                                                                                                \
        if (f16) FFMOE_GEMVM(A, true, Y, true);                                                         \
        else if (wide_x) FFMOE_GEMVM(A, true, Y, false);                                                \
        else FFMOE_GEMVM(A, false, Y, false);                                                           \
    } while (0)
        if (wide_w) { if (y_f32) FFMOE_GEMVM_X(true, true); else FFMOE_GEMVM_X(true, false); }
        else { if (y_f32) FFMOE_GEMVM_X(false, true); else FFMOE_GEMVM_X(false, false); }
#undef FFMOE_GEMVM_X
#undef FFMOE_GEMVM
        return hipGetLastError();
    }
    const uint32_t waves = (m + kRowsPerWave - 1) / kRowsPerWave;
    const dim3 grid((waves + 3) / 4), block(256);
    const bool aligned = (reinterpret_cast<uintptr_t>(w) % 16 == 0) && ((n / 2) % 16 == 0);
    const bool x_aligned = (reinterpret_cast<uintptr_t>(x) % 16 == 0) && (x_stride % 8 == 0);
#define FFMOE_GEMV16(A, F) \
    hipLaunchKernelGGL((gemv_int4_kernel<A, true, F, true>), grid, block, 0, s, w, scales, biases, x, y, m, n, rows, x_stride, y_stride, ids)
    if (f16) {
        if (!x_aligned) return hipErrorInvalidValue;     // FP16 rows come 16-byte aligned (checked at the boundary)
        if (aligned) { if (y_f32) FFMOE_GEMV16(true, true); else FFMOE_GEMV16(true, false); }
        else { if (y_f32) FFMOE_GEMV16(false, true); else FFMOE_GEMV16(false, false); }
        return hipGetLastError();
    }
#undef FFMOE_GEMV16
#define FFMOE_GEMV(A, X, F) \
    hipLaunchKernelGGL((gemv_int4_kernel<A, X, F, false>), grid, block, 0, s, w, scales, biases, x, y, m, n, rows, x_stride, y_stride, ids)
    if (aligned && x_aligned) { if (y_f32) FFMOE_GEMV(true, true, true); else FFMOE_GEMV(true, true, false); }
    else if (aligned) { if (y_f32) FFMOE_GEMV(true, false, true); else FFMOE_GEMV(true, false, false); }
    else if (x_aligned) { if (y_f32) FFMOE_GEMV(false, true, true); else FFMOE_GEMV(false, true, false); }
    else { if (y_f32) FFMOE_GEMV(false, false, true); else FFMOE_GEMV(false, false, false); }
#undef FFMOE_GEMV
    return hipGetLastError();
}

}  // namespace ffmoe
