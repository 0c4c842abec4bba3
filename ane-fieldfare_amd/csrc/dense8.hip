// The 8-bit dense FFN at many rows (Metal/Quant's 8-bit affine matrices as the packs hold the shared expert): two GEMMs on the
// matrix unit over integer operands.
//
// A weight is w = q s + b with q in 0..255, s and b per row and 64-wide group. q is exact in bf16 and in FP16, so a group's
// sum over q x runs on the matrix unit as it is and enters the running sum as s * sum - one fma per element and group - with
// no rounding of a weight. What the biases add is one more product of the same shape, sum_g b_g * (sum of x over group g):
// b is a bf16 value, the group sums are split into three bf16 values each (24 significant bits), and the three columns per
// group stand behind K as "groups" of scale 1. The alternative that keeps 16-bit weights to the same accuracy, hi and lo
// halves of every weight, doubles the products (matrix.hip keeps that form for the row counts at which it is still the faster one).
//
// Layouts: operands in matrix-instruction order, a fragment = 64 lanes x 16 bytes. Inputs: [16-row block][group][k-half][lane],
// lane (j, jq) = row j of the block, k = 32 * (k-half) + 8 * jq .. + 7 of the group. Weights: [128-row block][group][16-row tile
// of it][k-half][lane], scales [128-row block][group][row j of a tile][tile]. The gated matrix alternates gate and up tiles.
#include "common.hpp"
#include "kernels.hpp"

namespace ffmoe {
namespace {

constexpr int kTilesN = 8;                                  // 16-row tiles per N-block
constexpr int kBFrags = kTilesN * 2;                        // weight fragments per N-block and group
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t ext_groups(uint32_t n_groups) { return (3 * n_groups + kGroup - 1) / kGroup; }

// Column c of the bias columns, row j of a 16-row block: where it stands behind the block's (or N-block tile's) groups.
__device__ __forceinline__ uint32_t ext_lane(uint32_t c, uint32_t j) { return ((c & 31) >> 3) * 16 + j; }

// a row's group sum as three bf16 values that add up to its 24 significant bits
__device__ __forceinline__ void split_sum(float s, uint16_t (&part)[3]) {
#pragma unroll
    for (int p = 0; p < 3; ++p) {
        part[p] = f32_to_bf16(s);
        s -= bf16_to_f32(part[p]);
    }
}

// Weights: from the nibble planes of the resident matrix (matrix.hip) to operands. One thread per 8 elements of a stored row.
template <bool F16>
__global__ __launch_bounds__(256) void dense8_weights_kernel(const uint8_t *__restrict__ tiles, const uint8_t *__restrict__ scales,
                                                             uint32_t n_tiles, uint32_t n_groups, uint16_t *__restrict__ out,
                                                             float *__restrict__ out_scale) {
    const uint32_t all_groups = n_groups + ext_groups(n_groups), n_blocks = (n_tiles + kTilesN - 1) / kTilesN;
    const size_t total = (size_t)n_blocks * kTilesN * 16 * all_groups * 8;
    for (size_t gid = (size_t)blockIdx.x * 256 + threadIdx.x; gid < total; gid += (size_t)gridDim.x * 256) {
        const uint32_t piece = (uint32_t)(gid & 7), grp = (uint32_t)(gid / 8 % all_groups), row = (uint32_t)(gid / 8 / all_groups);
        const uint32_t tr = row >> 4, i = row & 15, jq = piece & 3, kh = piece >> 2;
        const bool real = tr < n_tiles;                     // tiles past the matrix (half an N-block): zeros
        uint32_t w[4] = {0, 0, 0, 0};
        float sc = 1.0f;                                    // the bias columns' scale
        if (grp < n_groups) {
            sc = 0.0f;
            if (real) {
                const size_t tile = (size_t)tr * n_groups + grp;
                const uint32_t *words = reinterpret_cast<const uint32_t *>(tiles + tile * kTileBytes) + (jq * 16 + i) * 4;
                const uint32_t high = words[kh], low = words[2 + kh];
                sc = bf16lo_to_f32(reinterpret_cast<const uint2 *>(scales + tile * kTileScaleBytes)[i].y);
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    const int pos = (t & 1) ? 4 + (t >> 1) : (t >> 1);          // arena order of the nibbles (common.hpp)
                    const float q = (float)(16u * ((high >> (4 * pos)) & 0xFu) + ((low >> (4 * pos)) & 0xFu));
                    w[t >> 1] |= (uint32_t)Act<F16>::round(q) << (16 * (t & 1));
                }
            }
        } else if (real) {
            const uint32_t c0 = (grp - n_groups) * kGroup + 32 * kh + 8 * jq;
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const uint32_t g = (c0 + t) / 3;
                if (g < n_groups) {
                    const uint32_t b = reinterpret_cast<const uint2 *>(scales + ((size_t)tr * n_groups + g) * kTileScaleBytes)[i].x >> 16;
                    w[t >> 1] |= b << (16 * (t & 1));
                }
            }
        }
        const size_t at = (size_t)(tr / kTilesN) * all_groups + grp;
        reinterpret_cast<uint4 *>(out)[(at * kBFrags + (tr % kTilesN) * 2 + kh) * kWave + jq * 16 + i] = uint4{w[0], w[1], w[2], w[3]};
        if (piece == 0) out_scale[(at * 16 + i) * kTilesN + tr % kTilesN] = sc;
    }
}

// Input rows to operands, with their group sums in the bias columns; rows past the last are zeros. One wave per 16-row block
// and group. The second GEMM's bias columns past its last group are cleared here too (its sums come from the first's epilogue).
template <bool F16>
__global__ __launch_bounds__(256) void dense8_rows_kernel(const uint16_t *__restrict__ x, uint32_t x_stride, uint32_t t, uint32_t n_groups,
                                                          uint16_t *__restrict__ out, uint32_t act_groups, uint16_t *__restrict__ acts) {
    const uint32_t lane = threadIdx.x & 63, j = lane & 15, jq = lane >> 4;
    const uint32_t item = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    const uint32_t block = item / n_groups, grp = item % n_groups, row = block * 16 + j;
    if (block * 16 >= t) return;
    const uint32_t all_groups = n_groups + ext_groups(n_groups);
    uint16_t *dst = out + (size_t)block * all_groups * 2 * (kWave * 8);
    float sum = 0.0f;
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
        const uint4 v = row < t ? *reinterpret_cast<const uint4 *>(x + (size_t)row * x_stride + grp * kGroup + 32 * kh + 8 * jq) : uint4{0, 0, 0, 0};
        reinterpret_cast<uint4 *>(dst)[(grp * 2 + kh) * kWave + lane] = v;
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) sum += Act<F16>::lo(w[q]) + Act<F16>::hi(w[q]);
    }
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    auto ext_at = [&](uint16_t *base, uint32_t first, uint32_t c) -> uint16_t & {
        return base[((size_t)(first + (c >> 6)) * 2 + ((c & 63) >> 5)) * (kWave * 8) + ext_lane(c, j) * 8 + (c & 7)];
    };
    if (jq == 0) {
        uint16_t part[3];
        split_sum(sum, part);
#pragma unroll
        for (int p = 0; p < 3; ++p) ext_at(dst, n_groups, 3 * grp + p) = part[p];
    }
    if (grp == 0) {
        for (uint32_t c = 3 * n_groups + jq; c < ext_groups(n_groups) * kGroup; c += 4) ext_at(dst, n_groups, c) = 0;
        uint16_t *adst = acts + (size_t)block * (act_groups + ext_groups(act_groups)) * 2 * (kWave * 8);
        for (uint32_t c = 3 * act_groups + jq; c < ext_groups(act_groups) * kGroup; c += 4) ext_at(adst, act_groups, c) = 0;
    }
}

// One block = 16 NMB (4 / WN) rows x one N-block of 128 weight rows; wave (wm, wn) owns every (4 / WN)th 16-row block from wm on
// and the tiles (8 / WN) wn ... Weights of a group (16 KiB) go through LDS in two buffers, a group ahead in registers; the inputs
// are in operand order and go straight to registers, a group ahead. Two fma of the tile before stand behind each product, so
// that the vector unit works in the matrix unit's shadow. GATED: out = the activations as the second GEMM's operands (with
// their group sums); else out = the output rows.
// Bound: the compute unit's LDS and load paths beside the matrix unit (at 128 rows and WN = 1, per group: 1,088 cycles of LDS
// for 512 of products on each SIMD; WN = 2 halves the fragment reads and loads every input twice, 218 us at 3,072 rows where
// WN = 1 takes 174). 3,072 rows of 2,816 -> 2,112 -> 2,816, whole FFN: 174-181 us against 248 for two library GEMMs on hi / lo
// rows with their epilogue passes. Measured and not kept: three groups of loads in flight (no change; two waves per SIMD
// fewer), 192-row tiles (178 us, and 251 against 206 at 4,096 rows, whose blocks they spread badly).
template <bool GATED, int NMB, int WN, bool F16>
__global__ __launch_bounds__(256, 2) void dense8_gemm_kernel(const uint16_t *__restrict__ weights, const float *__restrict__ scales,
                                                             uint32_t n_groups, uint32_t n_blocks, uint32_t n_cols,
                                                             const uint16_t *__restrict__ a, uint32_t t, uint16_t *__restrict__ out,
                                                             uint32_t out_stride) {
    __shared__ __align__(16) uint4 wb[2][kBFrags * kWave];
    __shared__ __align__(16) float sb[2][16 * kTilesN];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), j = lane & 15, jq = lane >> 4;
    constexpr int WM = 4 / WN;                              // waves side by side over the rows, over the tiles
    const uint32_t wm = wave % WM, wn = wave / WM;
    // all row tiles of an N-block on one XCD: its weights are read into one L2
    const uint32_t xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, per_xcd = (n_blocks + 7) / 8;
    const uint32_t mt = slot / per_xcd, nb = (slot % per_xcd) * 8 + xcd;
    if (nb >= n_blocks) return;
    const uint32_t ge = ext_groups(n_groups), all_groups = n_groups + ge, row_blocks = (t + 15) / 16;
    const u32x4_t *wsrc = reinterpret_cast<const u32x4_t *>(weights) + (size_t)nb * all_groups * (kBFrags * kWave) + tid;
    const float *ssrc = scales + (size_t)nb * all_groups * (16 * kTilesN) + (tid & 127);
    const uint4 *asrc[NMB];
    uint32_t blk[NMB];
#pragma unroll
    for (int i = 0; i < NMB; ++i) {
        blk[i] = mt * (WM * NMB) + wm + WM * i;
        // blocks past the last read it again (never stored)
        asrc[i] = reinterpret_cast<const uint4 *>(a) + (size_t)min(blk[i], row_blocks - 1) * all_groups * (2 * kWave) + lane;
    }
    const uint32_t last = all_groups - 1;                   // loads past the end fetch the last group again, never used
    u32x4_t wst[4];
    float sst = 0.0f;
    auto load_b = [&](uint32_t grp) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < 4; ++k) wst[k] = wsrc[(size_t)grp * (kBFrags * kWave) + 256 * k];
        sst = ssrc[grp * (16 * kTilesN)];
    };
    auto store_b = [&](uint32_t buf) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < 4; ++k) reinterpret_cast<u32x4_t *>(wb[buf])[256 * k + tid] = wst[k];
        if (tid < 16 * kTilesN) sb[buf][tid] = sst;
    };
    uint4 an[NMB][2];
    auto load_a = [&](uint32_t grp) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NMB; ++i)
#pragma unroll
            for (int kh = 0; kh < 2; ++kh) an[i][kh] = asrc[i][(grp * 2 + kh) * kWave];
    };
    constexpr int kTiles = kTilesN / WN;                    // of this wave
    f32x4 tot[NMB][kTiles];
#pragma unroll
    for (int i = 0; i < NMB; ++i)
#pragma unroll
        for (int nf = 0; nf < kTiles; ++nf) tot[i][nf] = f32x4{0.f, 0.f, 0.f, 0.f};

    // H: the element type of this group's operands (the bias columns are bf16 in either mode)
    auto step = [&](uint32_t grp, auto type) __attribute__((always_inline)) {
        constexpr bool H = decltype(type)::value;
        const uint32_t buf = grp & 1;
        uint4 af[NMB][2];
#pragma unroll
        for (int i = 0; i < NMB; ++i) af[i][0] = an[i][0], af[i][1] = an[i][1];
        store_b(buf ^ 1);                                   // group grp + 1 (past the last: a buffer nobody reads)
        load_b(min(grp + 2, last));
        load_a(min(grp + 1, last));
        float sc[kTiles];
#pragma unroll
        for (int nf = 0; nf < kTiles; nf += 4) {
            const f32x4 v = *reinterpret_cast<const f32x4 *>(&sb[buf][j * kTilesN + kTiles * wn + nf]);
            sc[nf] = v[0], sc[nf + 1] = v[1], sc[nf + 2] = v[2], sc[nf + 3] = v[3];
        }
        // tile by tile: its products, and the sums of the tile before between them, two fma behind each product
        // (a wave alone on its SIMD asks for all its fragments first: their latency is then paid once per group)
        constexpr int kQueue = WN == 2 ? kTiles : 2;
        uint4 bq[kQueue][2];
        auto read_b = [&](int nf) __attribute__((always_inline)) {
#pragma unroll
            for (int kh = 0; kh < 2; ++kh) bq[nf % kQueue][kh] = wb[buf][((kTiles * wn + nf) * 2 + kh) * kWave + lane];
        };
        f32x4 part[2][NMB];
        auto add = [&](int nf, int f) __attribute__((always_inline)) {
            tot[f >> 2][nf][f & 3] = __builtin_fmaf(sc[nf], part[nf & 1][f >> 2][f & 3], tot[f >> 2][nf][f & 3]);
        };
#pragma unroll
        for (int nf = 0; nf < kQueue - 1; ++nf) read_b(nf);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int nf = 0; nf < kTiles; ++nf) {
            if (nf + kQueue - 1 < kTiles) read_b(nf + kQueue - 1);
#pragma unroll
            for (int m = 0; m < 2 * NMB; ++m) {
                const int i = m % NMB, kh = m / NMB;
                const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
                part[nf & 1][i] = Act<H>::mfma(af[i][kh], bq[nf % kQueue][kh], kh ? part[nf & 1][i] : zero);
                if (nf > 0) {
                    add(nf - 1, 2 * m);
                    add(nf - 1, 2 * m + 1);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int f = 0; f < 4 * NMB; ++f) add(kTiles - 1, f);
        lds_barrier();
    };
    load_b(0);
    load_a(0);
    store_b(0);
    load_b(min(1u, last));
    lds_barrier();
    for (uint32_t grp = 0; grp < n_groups; ++grp) step(grp, std::integral_constant<bool, F16>{});
    for (uint32_t grp = n_groups; grp < all_groups; ++grp) step(grp, std::integral_constant<bool, false>{});

    // lane (j, jq) holds weight row j of every tile for rows 4 jq .. 4 jq + 3 of every 16-row block; each wave turns its blocks
    // through a piece of the weight buffers of its own (the last step ended with a barrier)
    constexpr uint32_t kStageRow = kTiles * 32 + 16;        // bytes: 64 columns + padding
    constexpr uint32_t kStageBytes = 4 * 16 * kStageRow, kRows = 16 * WM * NMB;
    static_assert(kStageBytes + 2 * kRows * sizeof(float) <= sizeof(wb), "staging and row sums fit the weight buffers");
    uint8_t *stage = reinterpret_cast<uint8_t *>(wb) + wave * 16 * kStageRow;
    float *row_sums = reinterpret_cast<float *>(reinterpret_cast<uint8_t *>(wb) + kStageBytes);      // [k-half][row of the tile]
    auto wave_sync = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    const uint32_t f_groups = n_blocks, f_all = f_groups + ext_groups(f_groups);         // (GATED: an N-block is a group of F)
#pragma unroll
    for (int i = 0; i < NMB; ++i) {
        if (blk[i] >= row_blocks) continue;                 // wave-uniform
        if constexpr (GATED) {
            // tiles 2 tl and 2 tl + 1 of this wave: gate and up of 16 activations; its share of group nb is k-half wn, or both
            uint16_t *img = reinterpret_cast<uint16_t *>(stage);
            float sum[2 / WN][4] = {};             // per k-half, so that both splits of the tiles add up alike
#pragma unroll
            for (int tl = 0; tl < kTiles / 2; ++tl)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float g = Act<F16>::widen(Act<F16>::round(tot[i][2 * tl][r])), u = Act<F16>::widen(Act<F16>::round(tot[i][2 * tl + 1][r]));
                    const uint16_t v = Act<F16>::round(gelu_tanh_fast(g) * u);
                    sum[tl >> 1][r] += Act<F16>::widen(v);
                    img[((tl >> 1) * kWave + ((tl & 1) * 2 + (j >> 3)) * 16 + 4 * jq + r) * 8 + (j & 7)] = v;
                }
#pragma unroll
            for (int h = 0; h < 2 / WN; ++h)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
#pragma unroll
                    for (int m = 1; m < 16; m <<= 1) sum[h][r] += __shfl_xor(sum[h][r], m, 64);
                    if (j == 0) row_sums[(wn + h) * kRows + (wm + WM * i) * 16 + 4 * jq + r] = sum[h][r];
                }
            wave_sync();
#pragma unroll
            for (int h = 0; h < 2 / WN; ++h)
                reinterpret_cast<uint4 *>(out)[(((size_t)blk[i] * f_all + nb) * 2 + wn + h) * kWave + lane] =
                    reinterpret_cast<const uint4 *>(stage)[h * kWave + lane];
            wave_sync();
        } else {
#pragma unroll
            for (int nf = 0; nf < kTiles; ++nf)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    *reinterpret_cast<uint16_t *>(stage + (4 * jq + r) * kStageRow + nf * 32 + 2 * j) = Act<F16>::round(tot[i][nf][r]);
            wave_sync();
#pragma unroll
            for (int p = 0; p < 4 / WN; ++p) {
                constexpr uint32_t kChunks = 2 * kTiles;                                 // 16-byte pieces of a staged row
                const uint32_t sub = (kWave / kChunks) * p + lane / kChunks, chunk = lane % kChunks, row = blk[i] * 16 + sub;
                const uint32_t col = nb * (kTilesN * 16) + wn * (kTiles * 16) + 8 * chunk;
                const uint4 v = *reinterpret_cast<const uint4 *>(stage + sub * kStageRow + 16 * chunk);
                if (row < t && col < n_cols) *reinterpret_cast<uint4 *>(out + (size_t)row * out_stride + col) = v;
            }
            wave_sync();
        }
    }
    if constexpr (GATED) {
        // the group sums of the activations as they were rounded, into the second GEMM's bias columns
        lds_barrier();
        const uint32_t block = mt * (WM * NMB) + (tid >> 4);
        if (tid < kRows && block < row_blocks) {
            uint16_t part[3];
            split_sum(row_sums[tid] + row_sums[kRows + tid], part);
            uint16_t *dst = out + (size_t)block * f_all * 2 * (kWave * 8);
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                const uint32_t c = 3 * nb + p;
                dst[((size_t)(f_groups + (c >> 6)) * 2 + ((c & 63) >> 5)) * (kWave * 8) + ext_lane(c, tid & 15) * 8 + (c & 7)] = part[p];
            }
        }
    }
}

uint32_t all_groups_of(uint32_t n) { return n / kGroup + (3 * (n / kGroup) + kGroup - 1) / kGroup; }
uint32_t n_blocks_of(uint32_t stored_rows) { return (stored_rows / 16 + kTilesN - 1) / kTilesN; }

}  // namespace

// While its blocks are fewer than the compute units hold, a GEMM here takes one block's chain of groups, 0.7 us each however few
// the rows (a group's round trip), where the library's two take 22 us and 12.5 us per 1,000 rows and 10^6 weights of a
// projection: the lines cross where rows * d f / 10^6 is 68 times the groups of both products less 2,000 (fitted at 18
// widths, GPU time). Library form | this one, us: 2,816 -> 2,112, 576 rows 65 | 67, 704 rows 76 | 70, 3,072 rows 248 | 178; 2,816
// -> 704, 640 rows 41 | 50, 896 rows 53 | 52; 1,024 -> 2,816, 704 rows 52 | 57, 896 rows 59 | 59, 1,024 rows 67 | 60; 2,816 -> 2,816,
// 576 rows 78 | 77; 512 -> 512, 640 rows 24 | 22. Not below 640 rows, where the forms meet at the widest, nor beyond 1,024, where
// the narrowest (2,816 -> 256, 38 | 47) still cross, but in a call that the library's own 41 us on the host bound.
uint32_t dense8_min_rows(uint32_t d, uint32_t f) {
    const uint32_t groups = all_groups_of(d) + all_groups_of(f);
    const uint64_t line = groups * 68ull <= 2000ull ? 0 : (groups * 68ull - 2000ull) * 1000000ull / ((uint64_t)d * f);
    return (uint32_t)(line < 640 ? 640 : line > 1024 ? 1024 : line);
}

size_t dense8_weight_bytes(uint32_t stored_rows, uint32_t n) {
    const size_t blocks = (size_t)n_blocks_of(stored_rows) * all_groups_of(n);
    return blocks * (kBFrags * kWave * sizeof(uint4) + 16 * kTilesN * sizeof(float));
}

size_t dense8_operand_bytes(uint32_t rows, uint32_t n) { return (size_t)((rows + 15) / 16) * all_groups_of(n) * (2 * kWave) * sizeof(uint4); }

hipError_t launch_dense8_weights(hipStream_t s, const uint8_t *tiles, const uint8_t *scales, uint32_t stored_rows, uint32_t n, void *out,
                                 bool f16) {
    const size_t blocks = (size_t)n_blocks_of(stored_rows) * all_groups_of(n), threads = blocks * kTilesN * 16 * 8;
    float *out_scale = reinterpret_cast<float *>(static_cast<uint8_t *>(out) + blocks * (kBFrags * kWave * sizeof(uint4)));
    const dim3 grid((uint32_t)min((size_t)65535 * 16, (threads + 255) / 256));
    hipLaunchKernelGGL((f16 ? dense8_weights_kernel<true> : dense8_weights_kernel<false>), grid, dim3(256), 0, s, tiles, scales,
                       stored_rows / 16, n / kGroup, static_cast<uint16_t *>(out), out_scale);
    return hipGetLastError();
}

hipError_t launch_dense8_rows(hipStream_t s, const uint16_t *x, uint32_t x_stride, uint32_t t, uint32_t d, uint32_t f, void *x_ops, void *act_ops,
                              bool f16) {
    const dim3 grid(((t + 15) / 16 * (d / kGroup) + 3) / 4);
    hipLaunchKernelGGL((f16 ? dense8_rows_kernel<true> : dense8_rows_kernel<false>), grid, dim3(256), 0, s, x, x_stride, t, d / kGroup,
                       static_cast<uint16_t *>(x_ops), f / kGroup, static_cast<uint16_t *>(act_ops));
    return hipGetLastError();
}

hipError_t launch_dense8_gemm(hipStream_t s, const void *weights, uint32_t stored_rows, uint32_t n, bool gated, const void *ops, uint32_t t,
                              void *out, uint32_t out_stride, bool f16, uint32_t n_cus) {
    const uint32_t n_blocks = n_blocks_of(stored_rows), row_blocks = (t + 15) / 16;
    const float *scales = reinterpret_cast<const float *>(static_cast<const uint8_t *>(weights) +
                                                          (size_t)n_blocks * all_groups_of(n) * (kBFrags * kWave * sizeof(uint4)));
    // Tiles of 64 rows while a compute unit holds few of them: 128-row tiles halve the weights' way through LDS but leave a
    // chip that is not full to fewer blocks. The line is drawn on the XCD that has the most N-blocks (all row tiles of one run
    // there), at blocks of 64 rows per compute unit: 3 for the gated product, 1.75 for the plain one. Whole FFN,
    // 64 | 128 rows per tile in both products, us: 2,816 -> 2,112 -> 2,816, 640 rows (1.6 and 0.9 blocks) 72 | 78, 1,024 rows
    // (2.5, 1.5) 88 | 91, 1,280 rows (3.1, 1.9) 114 | 94, 3,072 rows 222 | 186; 2,816 -> 704, 1,024 rows (1, 1.5) 52 | 61, 2,048
    // rows (2, 3) 66 | 67; 704 -> 2,816, 1,152 rows (3.4, 0.6) 63 | 66, and 58 with 128 gated and 64 plain; 512 -> 512, 2,048
    // rows (1, 1) 26 | 30. Either gives the same bits.
    const uint32_t m64 = (row_blocks + 3) / 4;
    const bool small = 4 * ((n_blocks + 7) / 8) * m64 <= (gated ? 12u : 7u) * (n_cus / 8);
    const uint32_t tile_blocks = small ? 4 : 8, m_tiles = (row_blocks + tile_blocks - 1) / tile_blocks;
    const dim3 grid(8 * ((n_blocks + 7) / 8) * m_tiles);
#define FFMOE_DENSE8(N, W)                                                                                                              \
    hipLaunchKernelGGL((gated ? (f16 ? dense8_gemm_kernel<true, N, W, true> : dense8_gemm_kernel<true, N, W, false>)                      \
                              : (f16 ? dense8_gemm_kernel<false, N, W, true> : dense8_gemm_kernel<false, N, W, false>)),                  \
                       grid, dim3(256), 0, s, static_cast<const uint16_t *>(weights), scales, n / kGroup, n_blocks, stored_rows,          \
                       static_cast<const uint16_t *>(ops), t, static_cast<uint16_t *>(out), out_stride)
    if (small) FFMOE_DENSE8(2, 2);
    else FFMOE_DENSE8(2, 1);
#undef FFMOE_DENSE8
    return hipGetLastError();
}

}  // namespace ffmoe
