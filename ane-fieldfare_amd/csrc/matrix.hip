// Resident INT4 matrix: a [M][N] weight in the reference's row-major layout is re-tiled once into
// two-stream tiles and then serves 1..16 input rows per call at streaming speed, with an optional
// greedy choice (argmax) over the outputs.
//
// Replaces the LM head of LMHeadChainInt4.encodeGreedyDecode / encodeGreedyRows
// (Kernels/Fusions/LMHeadChainInt4.swift:94-139,225-284; Metal/Sampling/logit.metal:614-720,952-1005) and the
// static-weight uses of DequantInt4GEMV.encodeRows (Kernels/Quant/DequantInt4GEMV.swift:72-182).
// A tile holds rows a = 32 p + l % 16 (stream A) and a + 16 (stream B) of one 64-wide group, in the
// same lane order as the expert arena, so the kernels share the expert path's register-ring code.
//
// An 8-bit affine weight (Metal/Quant/dequant_int8.metal:5-12: w = q s + b, q = 0 .. 255) rides the same kernels as two
// 4-bit ones: q = 16 h + l, so w = (16 s) h + b + s l. A tile then holds rows 16 p + l % 16 twice - stream A their
// high nibbles with scale 16 s (exact: a power of two) and bias b, stream B their low nibbles with scale s and bias
// 0 - and an output is the sum of its two streams. Same bytes as the 8-bit matrix, same stream, same speed.
#include <cfloat>

#include "common.hpp"
#include "kernels.hpp"
#include "stream.hpp"
#include "topk.hpp"

namespace ffmoe {
namespace {

__device__ __forceinline__ uint32_t ref_nibbles8(const uint8_t *row, uint32_t k0) {
    const uint8_t *p = row + (k0 >> 1);
    return (uint32_t)p[0] | ((uint32_t)p[1] << 8) | ((uint32_t)p[2] << 16) | ((uint32_t)p[3] << 24);
}

// reference order (nibble j = element j) -> arena order (position m = element 2m, m + 4 = element 2m + 1)
__device__ __forceinline__ uint32_t to_arena_order(uint32_t v) {
    uint32_t out = 0;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        out |= ((v >> (8 * m)) & 0xFu) << (4 * m);
        out |= ((v >> (8 * m + 4)) & 0xFu) << (4 * m + 16);
    }
    return out;
}

__device__ __forceinline__ uint16_t load_u16(const uint8_t *p) { return (uint16_t)(p[0] | ((uint16_t)p[1] << 8)); }

// One thread per (tile, lane). Rows past M (M is padded up to a multiple of 32) become zero weights
// with zero scale and bias.
__global__ __launch_bounds__(256) void repack_matrix_kernel(const uint8_t *__restrict__ w, const uint8_t *__restrict__ s,
                                                            const uint8_t *__restrict__ b, uint32_t m, uint32_t n,
                                                            uint8_t *__restrict__ tiles, uint8_t *__restrict__ scales) {
    const uint32_t n_groups = n / kGroup, row_bytes = n / 2;
    const size_t n_tiles = (size_t)((m + 31) / 32) * n_groups;
    const size_t total = n_tiles * kWave;
    for (size_t gid = (size_t)blockIdx.x * blockDim.x + threadIdx.x; gid < total;
         gid += (size_t)gridDim.x * blockDim.x) {
        const uint32_t lane = gid & 63, i = lane & 15, jq = lane >> 4;
        const size_t tile = gid >> 6;
        const uint32_t rbp = tile / n_groups, grp = tile % n_groups;
        const uint32_t row_a = rbp * 2 * kTileRows + i, row_b = row_a + kTileRows;
        const uint32_t k0 = grp * kGroup + 8 * jq;
        uint4 chunk = {0, 0, 0, 0};
        if (row_a < m) {
            chunk.x = to_arena_order(ref_nibbles8(w + (size_t)row_a * row_bytes, k0));
            chunk.y = to_arena_order(ref_nibbles8(w + (size_t)row_a * row_bytes, k0 + 32));
        }
        if (row_b < m) {
            chunk.z = to_arena_order(ref_nibbles8(w + (size_t)row_b * row_bytes, k0));
            chunk.w = to_arena_order(ref_nibbles8(w + (size_t)row_b * row_bytes, k0 + 32));
        }
        reinterpret_cast<uint4 *>(tiles + tile * kTileBytes)[lane] = chunk;
        if (jq == 0) {
            uint2 sc = {0, 0};
            const size_t ia = ((size_t)row_a * n_groups + grp) * 2, ib = ((size_t)row_b * n_groups + grp) * 2;
            if (row_a < m) sc.x = (uint32_t)load_u16(s + ia) | ((uint32_t)load_u16(b + ia) << 16);
            if (row_b < m) sc.y = (uint32_t)load_u16(s + ib) | ((uint32_t)load_u16(b + ib) << 16);
            reinterpret_cast<uint2 *>(scales + tile * kTileScaleBytes)[i] = sc;
        }
    }
}

// The 8-bit form: w uint8 [m][n]. One thread per (tile, lane); a tile = 16 rows x one group, both nibble planes.
__device__ __forceinline__ void nibble_planes8(const uint8_t *p, uint32_t &high, uint32_t &low) {
    high = low = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        high |= (uint32_t)(p[i] >> 4) << (4 * i);
        low |= (uint32_t)(p[i] & 15u) << (4 * i);
    }
}

__global__ __launch_bounds__(256) void repack_matrix8_kernel(const uint8_t *__restrict__ w, const uint8_t *__restrict__ s,
                                                             const uint8_t *__restrict__ b, uint32_t m, uint32_t n,
                                                             uint8_t *__restrict__ tiles, uint8_t *__restrict__ scales) {
    const uint32_t n_groups = n / kGroup;
    const size_t n_tiles = (size_t)((m + 15) / 16) * n_groups;
    const size_t total = n_tiles * kWave;
    for (size_t gid = (size_t)blockIdx.x * blockDim.x + threadIdx.x; gid < total;
         gid += (size_t)gridDim.x * blockDim.x) {
        const uint32_t lane = gid & 63, i = lane & 15, jq = lane >> 4;
        const size_t tile = gid >> 6;
        const uint32_t rb = tile / n_groups, grp = tile % n_groups;
        const uint32_t row = rb * kTileRows + i, k0 = grp * kGroup + 8 * jq;
        uint4 chunk = {0, 0, 0, 0};
        if (row < m) {
            uint32_t h0, l0, h1, l1;
            nibble_planes8(w + (size_t)row * n + k0, h0, l0);
            nibble_planes8(w + (size_t)row * n + k0 + 32, h1, l1);
            chunk = uint4{to_arena_order(h0), to_arena_order(h1), to_arena_order(l0), to_arena_order(l1)};
        }
        reinterpret_cast<uint4 *>(tiles + tile * kTileBytes)[lane] = chunk;
        if (jq == 0) {
            uint2 sc = {0, 0};
            if (row < m) {
                const size_t at = ((size_t)row * n_groups + grp) * 2;
                const uint16_t scale = load_u16(s + at), bias = load_u16(b + at);
                sc.x = (uint32_t)f32_to_bf16(bf16_to_f32(scale) * 16.0f) | ((uint32_t)bias << 16);
                sc.y = (uint32_t)scale;
            }
            reinterpret_cast<uint2 *>(scales + tile * kTileScaleBytes)[i] = sc;
        }
    }
}

// Eight bytes of an 8-bit matrix's scales (16 s and b, s and 0) per thread.
__global__ __launch_bounds__(256) void large_scales8_kernel(const uint2 *__restrict__ scales, size_t count, uint32_t *__restrict__ large) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < count && (scales[i].y & 0x7FFFu) >= kLargeScale) *large = 1;
}

// Greedy choice per row: the largest finite value wins, ties go to the lowest index, NaN and +-inf never
// win; a row with no candidate yields index 0 (Metal/Sampling/logit.metal:689-720, 916-921). Two stages: the
// GEMV's blocks each leave the winner of the weight rows they walked, then one block per input row picks
// among those. A key orders by value first and by lower index second, so the order of comparisons is free.
__device__ __forceinline__ unsigned long long argmax_key(float v, uint32_t i) {
    if (!(__builtin_fabsf(v) < INFINITY)) return 0ull;       // NaN or +-inf: never chosen
    const uint32_t u = __float_as_uint(v);
    const uint32_t ord = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
    return ((unsigned long long)ord << 32) | (0xFFFFFFFFu - i);
}

// The winner's probability under the final logit softcap, as argmax_rows_f32 leaves it for a drafter
// (Metal/Sampling/logit.metal:946-1010): softmax over the finite logits, each capped to softcap * tanh(v / softcap)
// when softcap > 0, kept as an online (maximum, sum of exp(c - maximum)) pair that merges associatively.
struct SoftmaxAcc {
    float m, s;      // m = -inf: nothing seen yet
};
// The divisions as reciprocals with a step of Newton's method each: 11 instructions for some 35, and no further off (the quotient's error is
// below a unit in its last place, the second product and sum round once). Every positive cap has a place: the reciprocal of one below 2^-128
// is held to a number (0 stays 0), and it is r that is doubled, not the cap, which may be the largest number there is.
__device__ __forceinline__ float capped(float v, float softcap) {
    if (!(softcap > 0.0f)) return v;
    // tanh z = 1 - 2 / (exp(2 z) + 1); from z = 40 on (and where v / softcap is no number any more) that is 1
    const float inv = fminf(1.0f / softcap, FLT_MAX);
    float z = fminf(fmaxf(v * inv, -40.0f), 40.0f);
    z = fminf(__builtin_fmaf(__builtin_fmaf(-z, softcap, v), inv, z), 40.0f);
    const float d = __expf(2.0f * z) + 1.0f;
    float r = __builtin_amdgcn_rcpf(d);
    r = __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r);
    return __builtin_fmaf(-softcap, r + r, softcap);
}
__device__ __forceinline__ void softmax_take(SoftmaxAcc &a, float v, float softcap) {
    if (!(__builtin_fabsf(v) < INFINITY)) return;          // non-finite logits take no part (they never win either)
    const float c = capped(v, softcap);
    if (c > a.m) {
        a.s = a.s * __expf(a.m - c) + 1.0f;                 // exp(-inf) = 0 covers the first value
        a.m = c;
    } else {
        a.s += __expf(c - a.m);
    }
}
__device__ __forceinline__ SoftmaxAcc softmax_merge(const SoftmaxAcc &a, const SoftmaxAcc &b) {
    const float m = fmaxf(a.m, b.m);
    if (m == -INFINITY) return SoftmaxAcc{-INFINITY, 0.0f};
    return SoftmaxAcc{m, a.s * __expf(a.m - m) + b.s * __expf(b.m - m)};
}
__device__ __forceinline__ SoftmaxAcc softmax_shuffle(const SoftmaxAcc &a, int mask) {
    return SoftmaxAcc{__shfl_xor(a.m, mask, 64), __shfl_xor(a.s, mask, 64)};
}

// y[r][m] = sum_g [ s_g * sum_k q_k x_k + b_g * sum_k x_k ] (moe.metal:323-378, logit.metal:614-667) for all
// input rows at once. grid = (blocks): every block takes each gridDim.x-th 32-row tile; its four waves split K
// (at most kRing groups each), keep their slice of the input rows in registers and refill the weight
// ring across tiles; per tile the partial sums meet in LDS, are added in wave order, and each wave
// stores a quarter of the input rows. GREEDY: nothing is stored per weight row; every lane keeps the best
// (value, index) key of the sums it finishes and the block leaves one key per input row in
// y_[row * gridDim.x + block], so the [rows][m] fp32 logits never travel to memory and back. CONF: the block also
// leaves the softmax pair of the sums it finished in conf_part[row * gridDim.x + block].
// PLANES8: the matrix is an 8-bit one stored as two nibble planes (above): a tile is 16 rows, an output the sum of its
// two streams.
// FEW (up to four input rows of the plain form): input row t is operand row 4 t, so that one of a lane's four sums is all there is to
// keep up, and each operand lane loads its own bytes: the lanes of a row ask for the same ones, there is nothing to turn through LDS.
// 1 row, us without | so: 16,384 x 1,408 6.7 | 5.9, 16,384 x 2,816 7.2 | 6.8, 262,144 x 2,816 76.5 | 74.9.
// ONCE: the matrix is more than the memory side's cache holds (kReadOnce); with it the last of those takes 66.6 (with the refills pinned and every
// gridDim.x-th tile 60.7, 6.8 TB/s).
// A block takes every gridDim.x-th tile (the gated form a range of pairs): what the chip reads and, above all, writes at a time lies together then. With
// a range each, 512 blocks write 128-byte pieces of 16 rows 2 KiB apart, which are few of the caches' channels: 262,144 x 2,816, fp32 logits, us with
// ranges | so: 1 row 62.9 | 60.7, 4 66.2 | 63.5, 8 70.9 | 67.2, 16 76.1 | 72.1, greedy with confidence, 1 row, 68.4 | 66.9 (stores to one small region 67; non-temporal or write-through ones, four tiles' at a time, or whole lines by half a wave
// per row change nothing).
template <bool Y_F32, bool F16, bool GREEDY = false, bool CONF = false, bool PLANES8 = false, int GLU = 0, bool FEW = false, bool ONCE = false>
__global__ __launch_bounds__(256, 2) void matrix_gemv_kernel(const uint8_t *__restrict__ tiles,
                                                             const uint8_t *__restrict__ scales, uint32_t m,
                                                             uint32_t n_groups, const uint16_t *__restrict__ x,
                                                             uint32_t x_stride, uint32_t rows, void *__restrict__ y_,
                                                             uint32_t y_stride, float2 *__restrict__ conf_part = nullptr,
                                                             float softcap = 0.0f) {
    constexpr int kSums = FEW ? 1 : 4;
    __shared__ float s_red[2][kKSplit][2 * kSums][64];
    static_assert(!FEW || !(GREEDY || PLANES8 || GLU), "few rows of the plain form");
    static_assert(!(PLANES8 && GREEDY), "the greedy choice is built for the 4-bit head only");
    static_assert((GLU == 1) ? PLANES8 : true, "tile pairs are the 8-bit planes' gated form");
    // GLU == 1: tiles 2 p and 2 p + 1 hold rows 16 p ... 16 p + 15 of a gate and of an up projection; a block takes whole
    // pairs, and `m` counts the outputs gelu_tanh(gate . x) * (up . x)
    const uint32_t n_tiles = GLU == 1 ? 2 * ((m + 15) / 16) : PLANES8 ? (m + 15) / 16 : (m + 31) / 32;
    uint32_t rb0 = blockIdx.x, rb1 = n_tiles, every = gridDim.x;
    if (GLU == 1) {
        split_range(n_tiles / 2, gridDim.x, blockIdx.x, rb0, rb1);
        rb0 *= 2, rb1 *= 2, every = 1;
    }
    if (rb0 >= rb1) {
        if (GREEDY && threadIdx.x < rows) reinterpret_cast<unsigned long long *>(y_)[(size_t)threadIdx.x * gridDim.x + blockIdx.x] = 0ull;
        if (CONF && threadIdx.x < rows) conf_part[(size_t)threadIdx.x * gridDim.x + blockIdx.x] = make_float2(-INFINITY, 0.0f);
        return;
    }
    const uint32_t lane = threadIdx.x & 63, ks = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t j = lane & 15, jq = lane >> 4;
    const uint32_t per = (n_groups + kKSplit - 1) / kKSplit;
    const uint32_t g0 = min(ks * per, n_groups), g1 = min(n_groups, g0 + per), ng = g1 - g0;
    const uint32_t g_last = g1 > g0 ? g1 - 1 : n_groups - 1;
    const TileSource src = make_tile_source(tiles, (size_t)n_tiles * n_groups * kTileBytes, scales,
                                            (size_t)n_tiles * n_groups * kTileScaleBytes);
    // 17 to 32 input rows of the plain 16-bit form: grid row 1 takes those past the 16th and reads the weights again, then from the caches
    if (!(Y_F32 || GREEDY || PLANES8 || GLU)) {
        x += (size_t)blockIdx.y * FFMOE_MAX_VERIFY_ROWS * x_stride;
        y_ = reinterpret_cast<uint16_t *>(y_) + (size_t)blockIdx.y * FFMOE_MAX_VERIFY_ROWS * y_stride;
        rows = min((uint32_t)FFMOE_MAX_VERIFY_ROWS, rows - blockIdx.y * FFMOE_MAX_VERIFY_ROWS);
    }
    WeightRing ring;
#pragma unroll
    for (int u = 0; u < kRing; ++u) ring_fill_here<ONCE>(ring, u, src, rb0 * n_groups + min(g0 + u, g_last), lane);
    // the input rows of this wave's K-slice: requested as 64-byte pieces (four lanes per row), then turned into the
    // operand layout - with 16 rows the operand layout itself would make every lane of every load a request of its own
    uint4 x0[kRing], x1[kRing];
    if constexpr (FEW) {
        load_few_rows(x, x_stride, rows, lane, KSlice{g0, ng, g_last}, x0, x1);
    } else {
        load_token_rows(x, x_stride, rows, lane, KSlice{g0, ng, g_last}, x0, x1);
        turn_token_rows(lane, x0, x1);
    }
    // per group: the sum of its inputs per token column, once for all the tile rows this wave walks
    f32x4 sx[kRing];
#pragma unroll
    for (int u = 0; u < kRing; ++u) sx[u] = group_input_sum<F16>(x0[u], x1[u]);
    const uint32_t my_row = FEW ? jq : 4 * jq + ks;        // the input row this lane finishes (FEW: a wave finishes one stream, waves 2 and 3 none)
    float *y32 = reinterpret_cast<float *>(y_);
    uint16_t *y16 = reinterpret_cast<uint16_t *>(y_);
    unsigned long long best = 0ull;
    SoftmaxAcc soft{-INFINITY, 0.0f};
    float gate_kept = 0.0f;

    uint32_t buf = 1;
    for (uint32_t rb = rb0; rb < rb1; rb += every) {
        const bool more = rb + every < rb1;
        const uint32_t next_row = (more ? rb + every : rb) * n_groups;
        const uint32_t fill_lane = more || (size_t)n_tiles * n_groups >= kNoLaneTiles ? lane : no_lane(lane);
        TwoStreamAcc tot;
        tot.a = f32x4{0.f, 0.f, 0.f, 0.f};
        tot.b = tot.a;
#pragma unroll
        for (int u = 0; u < kRing; ++u)
            ring_step<F16, true, kSums, ONCE>(ring, u, (uint32_t)u < ng, x0[u], x1[u], sx[u], tot, src, next_row + min(g0 + u, g_last), fill_lane);
        buf ^= 1u;
#pragma unroll
        for (int r = 0; r < kSums; ++r) {
            s_red[buf][ks][r][lane] = tot.a[r];
            s_red[buf][ks][kSums + r][lane] = tot.b[r];
        }
        lds_barrier();
        if constexpr (FEW) {
            if (ks > 1) continue;
            float v = s_red[buf][0][ks][lane];
#pragma unroll
            for (int o = 1; o < kKSplit; ++o) v += s_red[buf][o][ks][lane];
            const uint32_t row = (rb * 2 + ks) * kTileRows + j;
            if (my_row < rows && row < m) {
                if (Y_F32) y32[(size_t)my_row * y_stride + row] = v;
                else y16[(size_t)my_row * y_stride + row] = Act<F16>::round(v);
            }
            continue;
        }
        float va = s_red[buf][0][ks][lane], vb = s_red[buf][0][4 + ks][lane];
#pragma unroll
        for (int o = 1; o < kKSplit; ++o) {
            va += s_red[buf][o][ks][lane];
            vb += s_red[buf][o][4 + ks][lane];
        }
        if (GLU == 1) {
            // both projections are rounded to 16 bits in front of the activation, as shared_int8_gate_up_act_simd does
            // (Metal/Quant/dequant_int8.metal:131-136) and as two separate calls with the activation between them would
            const float v = Act<F16>::widen(Act<F16>::round(va + vb));
            const uint32_t col = (rb >> 1) * kTileRows + j;
            if (!(rb & 1u)) {
                gate_kept = v;
            } else if (my_row < rows && col < m) {
                const float act = gelu_tanh_fast(gate_kept) * v;
                if (Y_F32) y32[(size_t)my_row * y_stride + col] = act;
                else y16[(size_t)my_row * y_stride + col] = Act<F16>::round(act);
            }
        } else if (PLANES8) {
            const uint32_t row = rb * kTileRows + j;
            if (my_row < rows && row < m) {
                const float v = va + vb;
                if (Y_F32) y32[(size_t)my_row * y_stride + row] = v;
                else y16[(size_t)my_row * y_stride + row] = Act<F16>::round(v);
            }
        } else if (my_row < rows) {
            const uint32_t row_a = rb * 2 * kTileRows + j, row_b = row_a + kTileRows;
            const size_t base = (size_t)my_row * y_stride;
            if (GREEDY) {
                const unsigned long long ka = row_a < m ? argmax_key(va, row_a) : 0ull;
                const unsigned long long kb = row_b < m ? argmax_key(vb, row_b) : 0ull;
                best = max(best, max(ka, kb));
                if (CONF) {
                    if (row_a < m) softmax_take(soft, va, softcap);
                    if (row_b < m) softmax_take(soft, vb, softcap);
                }
            } else if (Y_F32) {
                if (row_a < m) y32[base + row_a] = va;
                if (row_b < m) y32[base + row_b] = vb;
            } else {
                if (row_a < m) y16[base + row_a] = Act<F16>::round(va);
                if (row_b < m) y16[base + row_b] = Act<F16>::round(vb);
            }
        }
    }
    if (GREEDY) {
        // the 16 lanes that share lane / 16 finished the same input row
#pragma unroll
        for (int mk = 8; mk >= 1; mk >>= 1) best = max(best, (unsigned long long)__shfl_xor(best, mk, 64));
        if (j == 0 && my_row < rows)
            reinterpret_cast<unsigned long long *>(y_)[(size_t)my_row * gridDim.x + blockIdx.x] = best;
        if (CONF) {
#pragma unroll
            for (int mk = 8; mk >= 1; mk >>= 1) soft = softmax_merge(soft, softmax_shuffle(soft, mk));
            if (j == 0 && my_row < rows) conf_part[(size_t)my_row * gridDim.x + blockIdx.x] = make_float2(soft.m, soft.s);
        }
    }
}

// The plain 4-bit form for matrices of few tiles: a block takes ONE of a tile's two streams, 16 weight rows, so that twice as many
// compute units share the steps and each wave issues half of them; what the GEMV keeps per group for the tiles to come is not kept.
// FEW as in the GEMV. Every sum has the GEMV's operands in its order, so an output's bits do not depend on the form.
// What bounds it: a launch (3.2 us with one step in it) and a round trip. Before, turning the inputs was 88 exchanges through LDS per wave
// and the eleven steps some 70 instructions each on one compute unit in six. 1,408 x 2,816, us back to back, the GEMV | so: 1 row 5.8 | 3.7,
// 16 rows 5.8 | 4.3; 8,192 x 2,816, 1 row 5.9 | 4.9.
template <bool Y_F32, bool F16, bool FEW>
__global__ __launch_bounds__(256, 2) void matrix_gemv_half_kernel(const uint8_t *__restrict__ tiles, const uint8_t *__restrict__ scales, uint32_t m,
                                                                  uint32_t n_groups, const uint16_t *__restrict__ x, uint32_t x_stride,
                                                                  uint32_t rows, void *__restrict__ y_, uint32_t y_stride) {
    constexpr int kSums = FEW ? 1 : 4;
    __shared__ float s_red[kKSplit][kSums][64];
    const uint32_t n_tiles = (m + 31) / 32;
    const uint32_t tile = (blockIdx.x >> 4) * 8 + (blockIdx.x & 7), half = blockIdx.x >> 3 & 1;      // (a tile's halves on one XCD)
    if (tile >= n_tiles) return;
    const uint32_t lane = threadIdx.x & 63, ks = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 15, jq = lane >> 4;
    const KSlice k = k_slice(n_groups, ks);
    const uint8_t *const my_tiles = tiles + (size_t)tile * n_groups * kTileBytes + lane * 16 + half * 8;
    const uint8_t *const my_scales = scales + (size_t)tile * n_groups * kTileScaleBytes + j * 8 + half * 4;
    uint2 w[kRing];
    uint32_t sb[kRing];
#pragma unroll
    for (int u = 0; u < kRing; ++u) {
        const uint32_t grp = min(k.g0 + u, k.g_last);
        w[u] = *reinterpret_cast<const uint2 *>(my_tiles + (size_t)grp * kTileBytes);
        sb[u] = *reinterpret_cast<const uint32_t *>(my_scales + (size_t)grp * kTileScaleBytes);
    }
    uint4 x0[kRing], x1[kRing];
    if constexpr (FEW) {
        load_few_rows(x, x_stride, rows, lane, k, x0, x1);
    } else {
        load_token_rows(x, x_stride, rows, lane, k, x0, x1);
        turn_token_rows(lane, x0, x1);
    }
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    float tot[kSums];
#pragma unroll
    for (int r = 0; r < kSums; ++r) tot[r] = 0.0f;
#pragma unroll
    for (int u = 0; u < kRing; ++u) {
        const uint32_t sc = (uint32_t)u < k.ng ? sb[u] : 0u;
        const f32x4 sx = group_input_sum<F16>(x0[u], x1[u]);
        f32x4 acc = Act<F16>::mfma(x0[u], unpack8_offset<F16>(w[u].x), zero);
        acc = Act<F16>::mfma(x1[u], unpack8_offset<F16>(w[u].y), acc);
        const float s = bf16lo_to_f32(sc), t = __builtin_fmaf(-Act<F16>::kOffset, s, bf16hi_to_f32(sc));
#pragma unroll
        for (int r = 0; r < kSums; ++r) {
            tot[r] = __builtin_fmaf(s, acc[r], tot[r]);
            tot[r] = __builtin_fmaf(t, sx[r], tot[r]);
        }
    }
#pragma unroll
    for (int r = 0; r < kSums; ++r) s_red[ks][r][lane] = tot[r];
    lds_barrier();
    if (FEW && ks != 0) return;
    const uint32_t r = FEW ? 0 : ks;
    float v = s_red[0][r][lane];
#pragma unroll
    for (int o = 1; o < kKSplit; ++o) v += s_red[o][r][lane];
    const uint32_t row = FEW ? jq : 4 * jq + ks, col = tile * 2 * kTileRows + half * kTileRows + j;
    if (row >= rows || col >= m) return;
    if (Y_F32) reinterpret_cast<float *>(y_)[(size_t)row * y_stride + col] = v;
    else reinterpret_cast<uint16_t *>(y_)[(size_t)row * y_stride + col] = Act<F16>::round(v);
}

// The same sums for more than 16 input rows, 16 R of them per block: there the GEMV's grid rows each read the weights and every
// block its input rows again. A block has 8 / PARTS tiles and PARTS parts of K, a wave one of each: it expands a tile's nibbles
// once for R blocks of rows. The rows of all parts and the waves' tiles go straight into LDS, a ring of chunks of one or two
// groups ahead (all scales at once: a load of them per group takes the address unit as long as one of a tile); rows in
// 128-byte lines whose 16-byte piece c lies at c ^ (row % 8), so that the sixteen rows of an operand fall on different
// banks. A part of K is one or two of the GEMV's slices of K: each is summed by itself and the four are added in its order, so
// that a row has the GEMV's bits.
// GLU == 2: a 4-bit tile's stream A holds 16 rows of a gate projection and its stream B the same rows of the up projection - the
// expert arena's gate/up tiles - and `m` counts the outputs gelu_tanh(gate . x) * (up . x), both sums fp32 in front of the
// activation as in the expert kernels (moe.metal:496). GLU == 1 and PLANES8 as in the GEMV.
// Four parts run two blocks per compute unit (four waves per SIMD, 128 registers, half the LDS, chunks of one group): what one block's
// chain waits for the other fills. With one: 37 rows 14.3 us for both launches, now 12.9; 160 rows 23.3 | 20.8, 301 rows 32.0 | 28.7; 8 bits 19.4
// | 16.9 and, 160 rows, 34.0 | 29.1. Two parts keep one: their chains are twice as long, their sums twice the registers.
// Bound: up to some 100 rows the chain of groups of one item (the barrier, the expansion,
// the products and their sums one behind the other), beyond that the products and the sums themselves, a third of the products
// being the inputs' own sums, which every wave makes anew. Kept out, as they change nothing: the sums between the products or
// behind six of them, with and without a raised wave priority. 2,816 -> 2,112 -> 2,816, 4 bits, us of gate/up + down with the GEMV's
// passes of 16 rows | now: 96 rows 14 + 11 | 10 + 9, 190 rows 25 + 17 | 16 + 11, 301 rows 37 + 23 | 22 + 13, 384 rows 44 + 29 | 25 +
// 17 (17 rows 7.7 + 5.8 | 7.5 + 6.7: wide down products of up to 32 keep the passes, launch_matrix_gemv); 8 bits, 17 rows 10.8 + 7.4 | 9.3
// + 6.8, 37 rows 11.5 + 11.1 | 11.6 + 8.5, 190 rows 34 + 29 | 25 + 16 (all with one block per unit).
constexpr int kBandWaves = 8, kBandMax = 5;
template <int PARTS, int R> struct Band {
    static constexpr int tiles = kBandWaves / PARTS, slices = kKSplit / PARTS;
    static constexpr int blocks = PARTS / 2;                                        // per compute unit: PARTS waves per SIMD
    static constexpr int groups = R <= 3 && blocks == 1 ? 2 : 1;                    // of a chunk
    static constexpr int scale_loads = (slices * kRing * kTileScaleBytes + 1023) / 1024;
    static constexpr uint32_t x_bytes = PARTS * R * 2048, group_bytes = x_bytes + kBandWaves * kTileBytes;
    static constexpr uint32_t scales_at = 0, ring_at = kBandWaves * scale_loads * 1024, chunk_bytes = groups * group_bytes;
    static constexpr int room = (int)((160 * 1024 / blocks - ring_at) / chunk_bytes), depth = room < 6 ? room : 6;
    static constexpr uint32_t bytes = ring_at + depth * chunk_bytes;
    static constexpr int x_loads = (2 * R + tiles - 1) / tiles, loads = groups * (x_loads + 1);     // per wave and chunk
};

template <bool F16, bool PLANES8, int GLU, int PARTS, int R>
__global__ __launch_bounds__(64 * kBandWaves, PARTS) void matrix_band_kernel(const uint8_t *__restrict__ tiles, const uint8_t *__restrict__ scales,
                                                                         uint32_t m, uint32_t n_groups, const uint16_t *__restrict__ x,
                                                                         uint32_t x_stride, uint32_t rows, uint16_t *__restrict__ y,
                                                                         uint32_t y_stride) {
    using B = Band<PARTS, R>;
    static_assert(B::depth >= 2, "a chunk in use and one on its way");
    static_assert(B::tiles * (kKSplit - B::slices) * R * 8 * kWave * sizeof(float) <= B::bytes, "the other parts' sums fit");
    __shared__ __align__(16) uint8_t lds[B::bytes];
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 15, jq = lane >> 4;
    const uint32_t unit = wave % B::tiles, part = wave / B::tiles;
    const uint32_t n_tiles = GLU == 1 ? 2 * ((m + 15) / 16) : (PLANES8 || GLU == 2) ? (m + 15) / 16 : (m + 31) / 32;
    // the items tile set by tile set, an eighth of the list per XCD: each reads its eighth of the weights into its L2 once
    const uint32_t bands = ((rows + 15) / 16 + R - 1) / R, all = bands * ((n_tiles + B::tiles - 1) / B::tiles);
    const uint32_t xcd = blockIdx.x & 7, item = (uint32_t)((uint64_t)all * xcd / 8) + (blockIdx.x >> 3);
    if (item >= (uint32_t)((uint64_t)all * (xcd + 1) / 8)) return;
    const uint32_t row0 = item % bands * (16 * R), tile = item / bands * B::tiles + unit;
    const size_t at = (size_t)min(tile, n_tiles - 1) * n_groups;              // (past the last tile the last again, not stored)
    const uint8_t *const w_tiles = tiles + at * kTileBytes, *const w_scales = scales + at * kTileScaleBytes;
    const uint32_t per = (n_groups + kKSplit - 1) / kKSplit, g0 = part * B::slices * per, steps = B::slices * per;
    // the scales of the part's groups (past the last group the last bytes again, not used)
    const uint32_t scales_lds = wave * (B::scale_loads * 1024);
#pragma unroll
    for (int k = 0; k < B::scale_loads; ++k)
        global_to_lds_16(w_scales, min(g0 * kTileScaleBytes + k * 1024 + lane * 16, n_groups * kTileScaleBytes - 16), lds_base + B::scales_at + scales_lds + k * 1024);
    const uint16_t *from[B::x_loads];
    uint32_t to[B::x_loads];
#pragma unroll
    for (int k = 0; k < B::x_loads; ++k) {
        // 8 rows x 128 bytes per load (what does not divide by the waves, the last piece twice; rows past the last, the last)
        const uint32_t piece = min(unit + B::tiles * k, 2u * R - 1), row = min(row0 + piece * 8 + (lane >> 3), rows - 1);
        from[k] = x + (size_t)row * x_stride + 8 * ((lane & 7) ^ (lane >> 3));
        to[k] = part * (R * 2048) + piece * 1024;
    }
    auto load = [&](uint32_t step, uint32_t slot) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < B::groups; ++c) {
            const uint32_t grp = min(g0 + step + c, n_groups - 1), base = lds_base + slot + c * B::group_bytes;      // (past the last: read, not used)
            global_to_lds_16(w_tiles + (size_t)grp * kTileBytes, lane * 16, base + B::x_bytes + wave * kTileBytes);
#pragma unroll
            for (int k = 0; k < B::x_loads; ++k) global_to_lds_16(from[k] + grp * kGroup, base + to[k]);
        }
    };
    TwoStreamAcc tot[B::slices][R];
    TwoStreamAcc sum[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
        sum[i].a = sum[i].b = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < B::slices; ++q) tot[q][i].a = tot[q][i].b = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const uint32_t x_at = part * (R * 2048) + j * 128 + 16 * (jq ^ (j & 7));
#pragma unroll
    for (int d = 0; d < B::depth - 1; ++d) load(d * B::groups, B::ring_at + d * B::chunk_bytes);
    uint32_t slot = B::ring_at, before = B::ring_at + (B::depth - 1) * B::chunk_bytes;
#pragma nounroll
    for (uint32_t s = 0; s < steps; s += B::groups) {
        ring_barrier<(B::depth - 2) * B::loads>();          // this chunk's loads are there, and nobody reads the one before any more
        load(s + (B::depth - 1) * B::groups, before);
#pragma unroll
        for (int c = 0; c < B::groups; ++c) {
            if (B::slices == 2 && s + c == per) {
#pragma unroll
                for (int i = 0; i < R; ++i) {
                    tot[0][i] = sum[i];
                    sum[i].a = sum[i].b = f32x4{0.f, 0.f, 0.f, 0.f};
                }
            }
            if (s + c >= steps || g0 + s + c >= n_groups) continue;        // wave-uniform: the last slices may be short
            const uint8_t *const here = lds + slot + c * B::group_bytes;
            const uint4 t = *reinterpret_cast<const uint4 *>(here + B::x_bytes + wave * kTileBytes + lane * 16);
            const uint2 sc = *reinterpret_cast<const uint2 *>(lds + B::scales_at + scales_lds + (s + c) * kTileScaleBytes + j * 8);
            const uint4 a0 = unpack8_offset<F16>(t.x), a1 = unpack8_offset<F16>(t.y), b0 = unpack8_offset<F16>(t.z), b1 = unpack8_offset<F16>(t.w);
            const float sa = bf16lo_to_f32(sc.x), ba = bf16hi_to_f32(sc.x), sb = bf16lo_to_f32(sc.y), bb = bf16hi_to_f32(sc.y);
            const float ta = __builtin_fmaf(-Act<F16>::kOffset, sa, ba), tb = __builtin_fmaf(-Act<F16>::kOffset, sb, bb);
            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < R; ++i) {
                const uint4 x0 = *reinterpret_cast<const uint4 *>(here + x_at + i * 2048), x1 = *reinterpret_cast<const uint4 *>(here + (x_at ^ 64) + i * 2048);
                const f32x4 sx = group_input_sum<F16>(x0, x1);
                const f32x4 acc_a = Act<F16>::mfma(x1, a1, Act<F16>::mfma(x0, a0, zero)), acc_b = Act<F16>::mfma(x1, b1, Act<F16>::mfma(x0, b0, zero));
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    sum[i].a[r] = __builtin_fmaf(ta, sx[r], __builtin_fmaf(sa, acc_a[r], sum[i].a[r]));
                    sum[i].b[r] = __builtin_fmaf(tb, sx[r], __builtin_fmaf(sb, acc_b[r], sum[i].b[r]));
                }
            }
        }
        before = slot;
        slot = slot + B::chunk_bytes == B::bytes ? B::ring_at : slot + B::chunk_bytes;
    }
#pragma unroll
    for (int i = 0; i < R; ++i) tot[B::slices - 1][i] = sum[i];
    vmem_barrier<0>();                                      // no load is on its way into what follows
    lds_barrier();
    // the later parts' slices to the first part's waves
    constexpr int kOthers = kKSplit - B::slices;
    float *const sums = reinterpret_cast<float *>(lds) + unit * (kOthers * R * 8 * kWave) + lane;
    if (part) {
#pragma unroll
        for (int q = 0; q < B::slices; ++q)
#pragma unroll
            for (int i = 0; i < R; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float *const to_q = sums + (((part - 1) * B::slices + q) * R + i) * (8 * kWave);
                    to_q[r * kWave] = tot[q][i].a[r];
                    to_q[(4 + r) * kWave] = tot[q][i].b[r];
                }
    }
    lds_barrier();
    if (!part) {
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float va = tot[0][i].a[r], vb = tot[0][i].b[r];
                if (B::slices == 2) va += tot[B::slices - 1][i].a[r], vb += tot[B::slices - 1][i].b[r];
#pragma unroll
                for (int q = 0; q < kOthers; ++q) {
                    va += sums[(q * R + i) * (8 * kWave) + r * kWave];
                    vb += sums[(q * R + i) * (8 * kWave) + (4 + r) * kWave];
                }
                const uint32_t row = row0 + i * 16 + 4 * jq + r;
                uint16_t *const yr = y + (size_t)row * y_stride;
                if (GLU == 1) {
                    // gate or up, rounded as the GEMV rounds them; the pair's other wave has the other
                    sums[i * (8 * kWave) + r * kWave] = Act<F16>::widen(Act<F16>::round(va + vb));
                } else if (row < rows && tile < n_tiles) {
                    if (GLU == 2) {
                        const uint32_t col = tile * kTileRows + j;
                        if (col < m) yr[col] = Act<F16>::round(gelu_tanh_fast(va) * vb);
                    } else if (PLANES8) {
                        const uint32_t col = tile * kTileRows + j;
                        if (col < m) yr[col] = Act<F16>::round(va + vb);
                    } else {
                        const uint32_t col = tile * 2 * kTileRows + j;
                        if (col < m) yr[col] = Act<F16>::round(va);
                        if (col + kTileRows < m) yr[col + kTileRows] = Act<F16>::round(vb);
                    }
                }
            }
    }
    if (GLU == 1) {
        lds_barrier();
        if (part || tile >= n_tiles) return;
        // both waves of a pair have both projections in reach: each finishes every other of its rows' blocks of 16
        const float *const gate = reinterpret_cast<const float *>(lds) + (unit & ~1u) * (kOthers * R * 8 * kWave) + lane, *const up = gate + kOthers * R * 8 * kWave;
        const uint32_t col = (tile >> 1) * kTileRows + j;
#pragma unroll
        for (int i = 0; i < R; ++i) {
            if ((i & 1) != (int)(unit & 1)) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t row = row0 + i * 16 + 4 * jq + r;
                const float act = gelu_tanh_fast(gate[i * (8 * kWave) + r * kWave]) * up[i * (8 * kWave) + r * kWave];
                if (row < rows && col < m) y[(size_t)row * y_stride + col] = Act<F16>::round(act);
            }
        }
    }
}

// The block's largest key and, if it is wanted, its softmax pair (the largest value first, then the sums relative to it; no NaN comes
// here), for the threads of its first wave: the others are told to leave. WAVES: 4 or 16; a wave's lanes hold all waves' several times over.
template <int WAVES>
__device__ __forceinline__ bool block_choice(unsigned long long &best, SoftmaxAcc &soft, bool conf, unsigned long long *s_k, float2 *s_p) {
    best = wave_max_key(best);
    if (conf) {
        const float m = wave_max_f32(soft.m);
        soft = SoftmaxAcc{m, wave_butterfly_sum(soft.m > -INFINITY ? soft.s * __expf(soft.m - m) : 0.0f)};
    }
    if ((threadIdx.x & 63) == 0) {
        s_k[threadIdx.x >> 6] = best;
        s_p[threadIdx.x >> 6] = make_float2(soft.m, soft.s);
    }
    __syncthreads();
    if (threadIdx.x >= 64) return false;
    const float2 own = s_p[threadIdx.x & (WAVES - 1)];
    best = wave_max_key(s_k[threadIdx.x & (WAVES - 1)]);
    if (conf) {
        const float m = wave_max_f32(own.x);
        soft = SoftmaxAcc{m, row_butterfly_sum<WAVES>(own.x > -INFINITY ? own.y * __expf(own.x - m) : 0.0f)};
    }
    return true;
}

// The winner's value from its key (argmax_key is a bijection on the finite values).
__device__ __forceinline__ float key_value(unsigned long long k) {
    const uint32_t ord = (uint32_t)(k >> 32);
    return __uint_as_float((ord & 0x80000000u) ? (ord & 0x7FFFFFFFu) : ~ord);
}

__device__ __forceinline__ float winner_confidence(unsigned long long best, const SoftmaxAcc &all, float softcap) {
    if (best == 0ull || !(all.s > 0.0f)) return 0.0f;
    return __expf(capped(key_value(best), softcap) - all.m) / all.s;
}

__global__ __launch_bounds__(256) void argmax_final_kernel(const unsigned long long *__restrict__ part, uint32_t n_seg,
                                                           uint32_t *__restrict__ out, const float2 *__restrict__ conf_part,
                                                           float softcap, float *__restrict__ out_conf) {
    __shared__ unsigned long long s_k[4];
    __shared__ float2 s_p[4];
    const uint32_t row = blockIdx.x;
    unsigned long long best = 0ull;
    SoftmaxAcc soft{-INFINITY, 0.0f};
    for (uint32_t i = threadIdx.x; i < n_seg; i += 256) {
        const unsigned long long k = part[(size_t)row * n_seg + i];
        best = k > best ? k : best;
        if (out_conf) {
            const float2 q = conf_part[(size_t)row * n_seg + i];
            soft = softmax_merge(soft, SoftmaxAcc{q.x, q.y});
        }
    }
    if (!block_choice<4>(best, soft, out_conf != nullptr, s_k, s_p) || threadIdx.x != 0) return;
    out[row] = best ? 0xFFFFFFFFu - (uint32_t)best : 0u;
    if (out_conf) out_conf[row] = winner_confidence(best, soft, softcap);
}

// argmax_rows_f32 (Metal/Sampling/logit.metal:946-1010): the greedy choice over rows of fp32 logits that are in
// memory already (the listed GEMV's output: a drafter's hot vocabulary): the largest finite value, ties to the lowest
// position, 0xFFFFFFFF and confidence 0 when no value is finite; and the winner's probability under the softcap.
// One block per row; rows of more than kArgmaxOneBlock values (`segments` given) one block per kSampleSegment values, whose
// winners argmax_merge_kernel joins. A thread requests eight values before it looks at the first, and adds their
// exponentials relative to the largest of the eight (value by value it was a chain of exponentials: 16 rows of 4,099 took
// 10.4 us with 256 threads each, 6.2 us so; 5.2 with waves that skip what lies past the row's end and reductions by register moves
// instead of through the LDS crossbar; 4.6 with caps that divide by reciprocals and one barrier for both reductions; one row of 512 3.3 -> 2.7,
// of 4,099 4.6 -> 3.8; 16 rows of 32,768 in segments: 4.0 + 2.6 us).
constexpr int kArgmaxThreads = 1024, kArgmaxBatch = 8;
constexpr uint32_t kArgmaxOneBlock = 8192;

template <int THREADS>
__global__ __launch_bounds__(THREADS) void argmax_rows_kernel(const float *__restrict__ logits, uint32_t stride, uint32_t count, uint32_t per_block,
                                                              float softcap, uint32_t *__restrict__ out, float *__restrict__ out_conf,
                                                              SampleSegment *__restrict__ segments) {
    __shared__ unsigned long long s_k[THREADS / 64];
    __shared__ float2 s_p[THREADS / 64];
    const float *row = logits + (size_t)blockIdx.x * stride;
    const uint32_t lo = blockIdx.y * per_block, hi = min(count, lo + per_block);
    unsigned long long best = 0ull;
    SoftmaxAcc soft{-INFINITY, 0.0f};
    for (uint32_t base = lo + threadIdx.x; base < hi; base += kArgmaxBatch * THREADS) {
        float v[kArgmaxBatch];
#pragma unroll
        for (int u = 0; u < kArgmaxBatch; ++u) v[u] = base + u * THREADS < hi ? row[base + u * THREADS] : NAN;
        // (a wave past the row's end skips what it does not have: the caps and exponentials are what a block of 1,024 threads spends its time on)
        const uint32_t wave_base = __builtin_amdgcn_readfirstlane(base & ~63u);
        float m = soft.m;
#pragma unroll
        for (int u = 0; u < kArgmaxBatch; ++u) {
            if (wave_base + u * THREADS >= hi) {
                v[u] = -INFINITY;
                continue;
            }
            const unsigned long long k = argmax_key(v[u], base + u * THREADS);
            best = k > best ? k : best;
            if (!out_conf) continue;
            v[u] = k ? capped(v[u], softcap) : -INFINITY;       // non-finite values take no part
            m = fmaxf(m, v[u]);
        }
        if (out_conf && m > -INFINITY) {
            float sum = soft.s * __expf(soft.m - m);            // exp(-inf) = 0: nothing seen before
#pragma unroll
            for (int u = 0; u < kArgmaxBatch; ++u)
                if (wave_base + u * THREADS < hi) sum += __expf(v[u] - m);
            soft = SoftmaxAcc{m, sum};
        }
    }
    if (!block_choice<THREADS / 64>(best, soft, out_conf != nullptr, s_k, s_p) || threadIdx.x != 0) return;
    if (segments) {
        SampleSegment seg{};
        seg.best = best;
        seg.top = soft.m;
        seg.sum = soft.s;
        segments[(size_t)blockIdx.x * kSampleMaxSegments + blockIdx.y] = seg;
        return;
    }
    out[blockIdx.x] = best ? 0xFFFFFFFFu - (uint32_t)best : 0xFFFFFFFFu;
    if (out_conf) out_conf[blockIdx.x] = winner_confidence(best, soft, softcap);
}

__global__ __launch_bounds__(256) void argmax_merge_kernel(const SampleSegment *__restrict__ segments, uint32_t n_seg, float softcap,
                                                           uint32_t *__restrict__ out, float *__restrict__ out_conf) {
    __shared__ unsigned long long s_k[4];
    __shared__ float2 s_p[4];
    SampleSegment mine{};
    mine.top = -INFINITY;
    if (threadIdx.x < n_seg) mine = segments[(size_t)blockIdx.x * kSampleMaxSegments + threadIdx.x];
    unsigned long long best = mine.best;
    SoftmaxAcc soft{mine.top, mine.sum};
    if (!block_choice<4>(best, soft, out_conf != nullptr, s_k, s_p) || threadIdx.x != 0) return;
    out[blockIdx.x] = best ? 0xFFFFFFFFu - (uint32_t)best : 0xFFFFFFFFu;
    if (out_conf) out_conf[blockIdx.x] = winner_confidence(best, soft, softcap);
}
static_assert(kSampleMaxSegments <= 256, "one segment per thread of argmax_merge_kernel");

}  // namespace

size_t matrix_tiles_bytes(uint32_t m, uint32_t n, bool planes8) {
    return (size_t)(planes8 ? (m + 15) / 16 : (m + 31) / 32) * (n / kGroup) * kTileBytes;
}
size_t matrix_scales_bytes(uint32_t m, uint32_t n, bool planes8) {
    return (size_t)(planes8 ? (m + 15) / 16 : (m + 31) / 32) * (n / kGroup) * kTileScaleBytes;
}
// Parts of K per block and 16-row blocks per band: the pair that costs least by what was measured, in units of 0.18 us. Four parts, two
// blocks per compute unit: a unit's first block takes 14 and 1.3 R per group of its chain, the second beside it 6 and 0.9 R. Two parts,
// one block, twice the chain: 12 and R + 0.7 per group. 2,816 -> 2 x 2,112 gated, then 2,112 -> 2,816 in the same shape, 4 bits, us at
// parts.blocks: 37 rows 4.1 12.9, 4.2 16.4; 64 rows 4.1 15.6, 4.2 16.6; 96 rows 4.1 18.1, 4.2 16.9; 160 rows 4.1 22.6, 4.2 21.5, 4.3
// 26.7; 240 rows 4.1 29.4, 4.2 30.1, 4.3 27.2, 2.3 35; 384 rows 4.2 41.7, 4.3 40.2, 2.4 42.2. Any gives the same bits.
struct BandShape {
    uint32_t parts, blocks;
    uint64_t cost;
};
static BandShape band_shape(uint32_t rows, uint32_t n_tiles, uint32_t n_groups, uint32_t n_cus) {
    const uint32_t row_blocks = (rows + 15) / 16, per = (n_groups + kKSplit - 1) / kKSplit;
    BandShape best = {2, kBandMax, ~0ull};
    for (uint32_t parts = 4; parts >= 2; parts -= 2)
        for (uint32_t r = parts == 4 ? 1 : 2; r <= (parts == 4 ? 3u : (uint32_t)kBandMax); ++r) {
            const uint32_t per_block = kBandWaves / parts, items = (row_blocks + r - 1) / r * ((n_tiles + per_block - 1) / per_block);
            const uint64_t on_each = (items + n_cus - 1) / n_cus;
            const uint64_t cost = parts == 4 ? (on_each + 1) / 2 * (14 + 13 * per * r / 10) + on_each / 2 * (6 + 9 * per * r / 10) : on_each * (12 + per * (20 * r + 14) / 10);
            if (cost < best.cost) best = BandShape{parts, r, cost};
        }
    return best;
}
// What a gated product d -> f and a plain one back take in bands, in the same units (0.18 us; two launches are some 24 more).
uint64_t band_pair_cost(uint32_t rows, uint32_t d, uint32_t f, bool planes8, uint32_t n_cus) {
    const uint32_t f_tiles = (f + 15) / 16;
    return band_shape(rows, planes8 ? 2 * f_tiles : f_tiles, d / kGroup, n_cus).cost +
           band_shape(rows, planes8 ? (d + 15) / 16 : (d + 31) / 32, f / kGroup, n_cus).cost;
}
bool matrix_shape_ok(uint32_t n) { return n % kGroup == 0 && (n / kGroup + kKSplit - 1) / kKSplit <= (uint32_t)kRing; }

hipError_t launch_matrix_repack(hipStream_t s, const uint8_t *w, const uint16_t *scales, const uint16_t *biases,
                                uint32_t m, uint32_t n, uint8_t *tiles_out, uint8_t *scales_out, bool planes8) {
    const size_t total = matrix_tiles_bytes(m, n, planes8) / kTileBytes * kWave;
    const uint32_t blocks = (uint32_t)min((size_t)65535 * 16, (total + 255) / 256);
    if (planes8)
        hipLaunchKernelGGL(repack_matrix8_kernel, dim3(blocks), dim3(256), 0, s, w, reinterpret_cast<const uint8_t *>(scales),
                           reinterpret_cast<const uint8_t *>(biases), m, n, tiles_out, scales_out);
    else
        hipLaunchKernelGGL(repack_matrix_kernel, dim3(blocks), dim3(256), 0, s, w, reinterpret_cast<const uint8_t *>(scales),
                           reinterpret_cast<const uint8_t *>(biases), m, n, tiles_out, scales_out);
    return hipGetLastError();
}

hipError_t launch_matrix8_large_scales(hipStream_t s, const uint8_t *a, size_t a_bytes, const uint8_t *b, size_t b_bytes, uint32_t *large) {
    const hipError_t e = hipMemsetAsync(large, 0, sizeof *large, s);
    if (e != hipSuccess) return e;
    for (int k = 0; k < 2; ++k) {
        const size_t count = (k ? b_bytes : a_bytes) / sizeof(uint2);
        hipLaunchKernelGGL(large_scales8_kernel, dim3((uint32_t)((count + 255) / 256)), dim3(256), 0, s, reinterpret_cast<const uint2 *>(k ? b : a), count, large);
    }
    return hipGetLastError();
}

hipError_t launch_matrix_gemv(hipStream_t s, const uint8_t *tiles, const uint8_t *scales, uint32_t m, uint32_t n,
                              const uint16_t *x, uint32_t x_stride, uint32_t rows, void *y, uint32_t y_stride,
                              bool y_f32, uint32_t n_cus, bool f16, bool planes8, int glu) {
    // glu: 0 plain, 1 the 8-bit planes' tile pairs, 2 a 4-bit tile's two streams as gate and up (m = the gated outputs; more than 16
    // rows: up to there such a matrix is an expert's and takes the expert kernels)
    if (glu == 2 && (planes8 || y_f32)) return hipErrorInvalidValue;
    const uint32_t n_tiles = (planes8 || glu == 2) ? (m + 15) / 16 : (m + 31) / 32;      // glu == 1: pairs of tiles
    if (rows == 0 || rows > (1u << 20) || (rows > FFMOE_MAX_VERIFY_ROWS ? y_f32 : glu == 2)) return hipErrorInvalidValue;
    const uint32_t all_tiles = glu == 1 ? 2 * n_tiles : n_tiles;
    // 17 to 32 rows of the plain 4-bit form: beyond 32 groups the GEMV's two grid rows, all of whose weights are on their way at once,
    // beat the band's chain of groups. Gate/up in a band, then down bands | GEMV, us at 17 rows: 2,816 columns out, K of
    // 1,600 12.0 | 12.4, 1,792 12.1 | 12.6, 2,112 12.8 | 12.6, 2,816 13.6 | 13.0; 1,024 out, 1,920 9.9 | 10.1; 512 out, 1,792 8.8 | 9.3, 2,816
    // 10.3 | 9.7.
    const bool twice = rows > FFMOE_MAX_VERIFY_ROWS && rows <= 2 * FFMOE_MAX_VERIFY_ROWS && glu == 0 && !planes8 && n / kGroup > 8 * kKSplit;
    if (rows > FFMOE_MAX_VERIFY_ROWS && !twice) {
        const BandShape shape = band_shape(rows, all_tiles, n / kGroup, n_cus);
        const uint32_t bands = ((rows + 15) / 16 + shape.blocks - 1) / shape.blocks, per_block = kBandWaves / shape.parts;
        const dim3 grid((bands * ((all_tiles + per_block - 1) / per_block) + 7) / 8 * 8);
        auto launch = [&](auto parts, auto blocks) {
            constexpr int P = decltype(parts)::value, N = decltype(blocks)::value;
            auto kernel = glu == 2   ? (f16 ? matrix_band_kernel<true, false, 2, P, N> : matrix_band_kernel<false, false, 2, P, N>)
                          : glu == 1 ? (f16 ? matrix_band_kernel<true, true, 1, P, N> : matrix_band_kernel<false, true, 1, P, N>)
                          : planes8  ? (f16 ? matrix_band_kernel<true, true, 0, P, N> : matrix_band_kernel<false, true, 0, P, N>)
                                     : (f16 ? matrix_band_kernel<true, false, 0, P, N> : matrix_band_kernel<false, false, 0, P, N>);
            hipLaunchKernelGGL(kernel, grid, dim3(64 * kBandWaves), 0, s, tiles, scales, m, n / kGroup, x, x_stride, rows,
                               static_cast<uint16_t *>(y), y_stride);
        };
#define FFMOE_BAND(P, N) launch(std::integral_constant<int, P>{}, std::integral_constant<int, N>{})
        switch (shape.parts * 8 + shape.blocks) {
            case 4 * 8 + 1: FFMOE_BAND(4, 1); break;
            case 4 * 8 + 2: FFMOE_BAND(4, 2); break;
            case 4 * 8 + 3: FFMOE_BAND(4, 3); break;
            case 2 * 8 + 2: FFMOE_BAND(2, 2); break;
            case 2 * 8 + 3: FFMOE_BAND(2, 3); break;
            case 2 * 8 + 4: FFMOE_BAND(2, 4); break;
            default: FFMOE_BAND(2, kBandMax); break;
        }
#undef FFMOE_BAND
        return hipGetLastError();
    }
    // Half a tile per block while those run at once: three such blocks per compute unit with few rows (135 registers), and, with the
    // inputs to be turned in every one of them, not many more than one otherwise. us back to back with whole tiles | halves, N = 2,816: 1
    // row, 8,192 out 5.9 | 4.9, 12,288 out 7.1 | 6.1 (12,320 in whole tiles of few rows 6.7), 16,384 out 6.8 | 7.4; 5 rows, 4,100 out 5.9 | 5.4, 5,632 out 5.7 |
    // 5.6, 8,200 out 6.8 | 7.2; 16 rows, 4,100 out 5.9 | 5.6, 5,632 out 5.8 | 5.9, 10,000 out 7.4 | 7.8.
    if (!planes8 && glu == 0 && rows <= FFMOE_MAX_VERIFY_ROWS && (rows <= 4 ? 2 * n_tiles <= 3 * n_cus : 8 * n_tiles <= 5 * n_cus)) {
        const dim3 halves((n_tiles + 7) / 8 * 16);
        auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, halves, dim3(256), 0, s, tiles, scales, m, n / kGroup, x, x_stride, rows, y, y_stride); };
        auto pick = [&](auto few) {
            constexpr bool FEW = decltype(few)::value;
            if (f16) { if (y_f32) launch(matrix_gemv_half_kernel<true, true, FEW>); else launch(matrix_gemv_half_kernel<false, true, FEW>); }
            else { if (y_f32) launch(matrix_gemv_half_kernel<true, false, FEW>); else launch(matrix_gemv_half_kernel<false, false, FEW>); }
        };
        if (rows <= 4) pick(std::true_type{}); else pick(std::false_type{});
        return hipGetLastError();
    }
    // (two grid rows: a multiple of 8 blocks per row keeps a tile on one XCD, blocks go to the XCDs round robin, and its L2 serves the
    // second; blocks past the tile count leave at once)
    const dim3 grid(twice ? (min(2 * n_cus, n_tiles) + 7) / 8 * 8 : min(2 * n_cus, n_tiles), twice ? 2 : 1);
#define FFMOE_MGEMV(Y, H, P, ...)                                                                                           \
    hipLaunchKernelGGL((matrix_gemv_kernel<Y, H, false, false, P, __VA_ARGS__>), grid, dim3(256), 0, s, tiles, scales, m, n / kGroup, x, x_stride, \
                       rows, y, y_stride)
    if (glu == 1) {
        if (f16) { if (y_f32) FFMOE_MGEMV(true, true, true, 1); else FFMOE_MGEMV(false, true, true, 1); }
        else { if (y_f32) FFMOE_MGEMV(true, false, true, 1); else FFMOE_MGEMV(false, false, true, 1); }
    } else {
        auto pick = [&](auto once) {
            constexpr bool O = decltype(once)::value;
            if (planes8) {
                if (f16) { if (y_f32) FFMOE_MGEMV(true, true, true, 0, false, O); else FFMOE_MGEMV(false, true, true, 0, false, O); }
                else { if (y_f32) FFMOE_MGEMV(true, false, true, 0, false, O); else FFMOE_MGEMV(false, false, true, 0, false, O); }
            } else if (rows <= 4) {
                if (f16) { if (y_f32) FFMOE_MGEMV(true, true, false, 0, true, O); else FFMOE_MGEMV(false, true, false, 0, true, O); }
                else { if (y_f32) FFMOE_MGEMV(true, false, false, 0, true, O); else FFMOE_MGEMV(false, false, false, 0, true, O); }
            } else {
                if (f16) { if (y_f32) FFMOE_MGEMV(true, true, false, 0, false, O); else FFMOE_MGEMV(false, true, false, 0, false, O); }
                else { if (y_f32) FFMOE_MGEMV(true, false, false, 0, false, O); else FFMOE_MGEMV(false, false, false, 0, false, O); }
            }
        };
        // Read once from the memory side's cache on; 4 bits with more than four input rows, which take longer over their bytes, from a sixteenth more
        // on. us without the hint | with, N = 2,112: 4 bits, 1 row, 270 MB 61.3 | 61.0, 277 MB 58.6 | 56.5, 338 MB 74.2 | 68.1; 16 rows, 270 MB 68.8 | 74.1,
        // 277 MB 67.1 | 68.7, 290 MB 74.4 | 73.9, 338 MB 88.8 | 84.3; 8 bits, 1 row, 259 MB 55.0 | 53.3, 277 MB 62.1 | 60.2, 16 rows, 259 MB 56.0 | 55.9, 277 MB
        // 65.9 | 65.8, 338 MB 86.6 | 81.1.
        const size_t once_from = planes8 || rows <= 4 ? kMemoryCacheBytes : kMemoryCacheBytes / 16 * 17;
        if (!twice && (size_t)n_tiles * (n / kGroup) * kTileBytes > once_from) pick(std::true_type{}); else pick(std::false_type{});
    }
#undef FFMOE_MGEMV
    return hipGetLastError();
}

// out = round16(gelu_tanh(gate) * up) per element of `rows` rows of `count` values: gelu_mul_fp16
// (Metal/Primitives/utility.metal:4-17), the step between the projections of the 8-bit shared expert
// (shared_int8_gate_up_act_simd rounds gate and up to 16 bits in front of it: Metal/Quant/dequant_int8.metal:131-136).
template <bool F16>
__global__ __launch_bounds__(256) void gelu_mul_kernel(const uint16_t *gate, uint32_t gate_stride, const uint16_t *up,
                                                       uint32_t up_stride, uint16_t *out, uint32_t out_stride, uint32_t count) {
    // no __restrict__: `out` may be `gate` or `up` itself (each element is read before it is written, by the same lane)
    const uint32_t row = blockIdx.y;
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < count; i += gridDim.x * 256) {
        const float g = Act<F16>::widen(gate[(size_t)row * gate_stride + i]), u = Act<F16>::widen(up[(size_t)row * up_stride + i]);
        out[(size_t)row * out_stride + i] = Act<F16>::round(gelu_tanh_fast(g) * u);
    }
}

hipError_t launch_gelu_mul(hipStream_t s, const uint16_t *gate, uint32_t gate_stride, const uint16_t *up, uint32_t up_stride,
                           uint16_t *out, uint32_t out_stride, uint32_t rows, uint32_t count, bool f16) {
    const dim3 grid(min(64u, (count + 255) / 256), rows);
    if (f16) hipLaunchKernelGGL(gelu_mul_kernel<true>, grid, dim3(256), 0, s, gate, gate_stride, up, up_stride, out, out_stride, count);
    else hipLaunchKernelGGL(gelu_mul_kernel<false>, grid, dim3(256), 0, s, gate, gate_stride, up, up_stride, out, out_stride, count);
    return hipGetLastError();
}

// Rows of the resident 4-bit matrix dequantised: out[i][k] = round16((q s + b) * out_scale) for weight row ids[i] (or
// the one row `token_id` when ids is null) - embed_lookup_int4 (Metal/Quant/dequant_int4.metal:53-73) on the re-tiled
// copy, so that tied embeddings need no second table. One thread per two words of a tile that lie together
// (lane 16 (k / 8 % 4) + row % 16, words 2 (row / 16 % 2) + (k / 32 % 2)), i.e. elements 8 jq ... + 7 of a group's halves, and the
// row's scale pair. What bounds it is the memory's rate in requests: a row's 32 bytes per group lie in four lines and its scales in a
// fifth. A thread per word asks for twice the requests and scale pairs of the same lines: 262,144 x 2,816, random ids of two tables in turn, us of
// a call so | now: 1,000 rows 6.9 | 6.3, 3,072 rows 18.35 | 17.4, 8,192 rows 46.3 | 41.7; up to 301 rows 3.4 either way. An id past the
// table gives a row of zeros.
template <bool F16>
__global__ __launch_bounds__(256) void matrix_rows_kernel(const uint8_t *__restrict__ tiles, const uint8_t *__restrict__ scales,
                                                          uint32_t m, uint32_t n_groups, const uint32_t *__restrict__ ids,
                                                          uint32_t token_id, float out_scale, uint16_t *__restrict__ out,
                                                          uint32_t out_stride) {
    const uint32_t r = ids ? ids[blockIdx.y] : token_id;
    for (uint32_t w = blockIdx.x * 256 + threadIdx.x; w < n_groups * 4; w += gridDim.x * 256) {
        const uint32_t grp = w >> 2, jq = w & 3;
        uint32_t packed[2][4] = {};
        if (r < m) {
            const size_t tile = (size_t)(r >> 5) * n_groups + grp;
            const uint32_t i = r & 15, half = (r >> 4) & 1;
            const uint2 words = reinterpret_cast<const uint2 *>(tiles + tile * kTileBytes)[(jq * 16 + i) * 2 + half];
            const uint32_t sb = reinterpret_cast<const uint32_t *>(scales + tile * kTileScaleBytes)[i * 2 + half];
            const float sc = bf16_to_f32((uint16_t)(sb & 0xFFFFu)), bi = bf16_to_f32((uint16_t)(sb >> 16));
#pragma unroll
            for (int hi = 0; hi < 2; ++hi) {
                const uint32_t word = hi ? words.y : words.x;
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    const int pos = (t & 1) ? 4 + (t >> 1) : (t >> 1);          // arena order: position p = element 2p, p + 4 = element 2p + 1
                    const float q = (float)((word >> (4 * pos)) & 0xFu);
                    const float v = (q * sc + bi) * out_scale;                  // q * sc is exact in fp32: the reference's expression
                    packed[hi][t >> 1] |= (uint32_t)Act<F16>::round(v) << (16 * (t & 1));
                }
            }
        }
        uint16_t *to = out + (size_t)blockIdx.y * out_stride + grp * kGroup + 8 * jq;
#pragma unroll
        for (int hi = 0; hi < 2; ++hi)
            *reinterpret_cast<uint4 *>(to + 32 * hi) = uint4{packed[hi][0], packed[hi][1], packed[hi][2], packed[hi][3]};
    }
}

hipError_t launch_matrix_rows(hipStream_t s, const uint8_t *tiles, const uint8_t *scales, uint32_t m, uint32_t n, const uint32_t *ids,
                              uint32_t token_id, uint32_t count, float out_scale, uint16_t *out, uint32_t out_stride, bool f16) {
    if (count == 0 || count > 65535u) return hipErrorInvalidValue;
    const dim3 grid(min(64u, (n / 16 + 255) / 256), count);
    if (f16)
        hipLaunchKernelGGL(matrix_rows_kernel<true>, grid, dim3(256), 0, s, tiles, scales, m, n / kGroup, ids, token_id, out_scale, out, out_stride);
    else
        hipLaunchKernelGGL(matrix_rows_kernel<false>, grid, dim3(256), 0, s, tiles, scales, m, n / kGroup, ids, token_id, out_scale, out, out_stride);
    return hipGetLastError();
}

// An 8-bit matrix for the library's dense GEMM, used beyond the row counts the streaming passes are good for: a 16-bit
// matrix element cannot hold w = q s + b of an 8-bit q, so w is written as two - hi = round16(w) and lo = round16(w - hi),
// together 16 (bf16) or 22 (FP16) significant bits of w - and the GEMM multiplies by both: out[r] = hi rows, out[rows + r]
// = lo rows ([2 m][n], row-major; the gated matrix: gate hi, gate lo, up hi, up lo, [4 f][n]). Read back from the nibble
// planes, so it can be made again when the activation type changes. One thread per 8 consecutive elements.
template <bool F16>
__global__ __launch_bounds__(256) void expand_planes8_kernel(const uint8_t *__restrict__ tiles, const uint8_t *__restrict__ scales,
                                                             uint32_t m, uint32_t n_groups, bool glu, uint16_t *__restrict__ out) {
    const uint32_t n = n_groups * kGroup, tile_rows = (glu ? 2u : 1u) * ((m + 15) / 16);
    const size_t total = (size_t)tile_rows * 16 * n_groups * 8;
    for (size_t gid = (size_t)blockIdx.x * 256 + threadIdx.x; gid < total; gid += (size_t)gridDim.x * 256) {
        const uint32_t w = (uint32_t)(gid % (n_groups * 8)), stored_row = (uint32_t)(gid / (n_groups * 8));
        const uint32_t grp = w >> 3, piece = w & 7, tr = stored_row >> 4, i = stored_row & 15;
        // the weight row this stored row is, and where its hi / lo rows go
        const uint32_t row = glu ? (tr >> 1) * 16 + i : stored_row;
        if (row >= m) continue;
        const size_t hi_row = glu ? ((tr & 1u) ? 2 * (size_t)m + row : row) : row, lo_row = hi_row + m;
        const size_t tile = (size_t)tr * n_groups + grp;
        const uint32_t jq = piece & 3, second = piece >> 2;
        const uint32_t *lane_words = reinterpret_cast<const uint32_t *>(tiles + tile * kTileBytes) + (jq * 16 + i) * 4;
        const uint32_t high = lane_words[second], low = lane_words[2 + second];
        const uint2 sb = reinterpret_cast<const uint2 *>(scales + tile * kTileScaleBytes)[i];
        const float sc = bf16_to_f32((uint16_t)(sb.y & 0xFFFFu)), bi = bf16_to_f32((uint16_t)(sb.x >> 16));
        uint32_t hi_w[4] = {0, 0, 0, 0}, lo_w[4] = {0, 0, 0, 0};
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const int pos = (t & 1) ? 4 + (t >> 1) : (t >> 1);
            const float q = (float)(16u * ((high >> (4 * pos)) & 0xFu) + ((low >> (4 * pos)) & 0xFu));
            const float v = q * sc + bi;                       // q * sc is exact in fp32 (8 + 8 bits): the reference's q s + b
            const uint16_t h = Act<F16>::round(v);
            hi_w[t >> 1] |= (uint32_t)h << (16 * (t & 1));
            lo_w[t >> 1] |= (uint32_t)Act<F16>::round(v - Act<F16>::widen(h)) << (16 * (t & 1));
        }
        *reinterpret_cast<uint4 *>(out + hi_row * n + grp * kGroup + 8 * piece) = uint4{hi_w[0], hi_w[1], hi_w[2], hi_w[3]};
        *reinterpret_cast<uint4 *>(out + lo_row * n + grp * kGroup + 8 * piece) = uint4{lo_w[0], lo_w[1], lo_w[2], lo_w[3]};
    }
}

hipError_t launch_expand_planes8(hipStream_t s, const uint8_t *tiles, const uint8_t *scales, uint32_t m, uint32_t n, bool glu,
                                 uint16_t *out, bool f16) {
    const size_t total = (size_t)(glu ? 2 : 1) * ((m + 15) / 16) * 16 * (n / 8);
    const dim3 grid((uint32_t)min((size_t)65535 * 16, (total + 255) / 256));
    if (f16) hipLaunchKernelGGL(expand_planes8_kernel<true>, grid, dim3(256), 0, s, tiles, scales, m, n / kGroup, glu, out);
    else hipLaunchKernelGGL(expand_planes8_kernel<false>, grid, dim3(256), 0, s, tiles, scales, m, n / kGroup, glu, out);
    return hipGetLastError();
}

// Behind the GEMMs on the hi / lo rows: a weight row's result is the sum of its two columns.
// gated: sums [rows][4 f] (gate hi, gate lo, up hi, up lo) -> act[r][j] = round16(gelu_tanh(round16(gate)) * round16(up)),
// the same roundings as the streaming form's epilogue. plain: sums [rows][2 d] -> y[r][i] = round16(hi + lo).
template <bool F16, bool GATED>
__global__ __launch_bounds__(256) void hilo_epilogue_kernel(const float *__restrict__ sums, uint32_t width, uint16_t *__restrict__ out,
                                                            uint32_t out_stride) {
    const float *row = sums + (size_t)blockIdx.y * width * (GATED ? 4 : 2);
    for (uint32_t j = blockIdx.x * 256 + threadIdx.x; j < width; j += gridDim.x * 256) {
        float v = row[j] + row[width + j];
        if (GATED) {
            const float g = Act<F16>::widen(Act<F16>::round(v));
            const float u = Act<F16>::widen(Act<F16>::round(row[2 * width + j] + row[3 * width + j]));
            v = gelu_tanh_fast(g) * u;
        }
        out[(size_t)blockIdx.y * out_stride + j] = Act<F16>::round(v);
    }
}

hipError_t launch_hilo_epilogue(hipStream_t s, const float *sums, uint32_t rows, uint32_t width, bool gated, uint16_t *out,
                                uint32_t out_stride, bool f16) {
    if (rows == 0 || rows > 65535u) return hipErrorInvalidValue;
    const dim3 grid(min(16u, (width + 255) / 256), rows);
#define FFMOE_HILO(H, G) hipLaunchKernelGGL((hilo_epilogue_kernel<H, G>), grid, dim3(256), 0, s, sums, width, out, out_stride)
    if (f16) { if (gated) FFMOE_HILO(true, true); else FFMOE_HILO(true, false); }
    else { if (gated) FFMOE_HILO(false, true); else FFMOE_HILO(false, false); }
#undef FFMOE_HILO
    return hipGetLastError();
}

// keys per input row that launch_matrix_greedy leaves between its two kernels
uint32_t greedy_segments(uint32_t m, uint32_t n_cus) { return min(2 * n_cus, (m + 31) / 32); }

// `partials`: [16][segments] keys, then (when out_conf is wanted) [16][segments] softmax pairs
hipError_t launch_matrix_greedy(hipStream_t s, const uint8_t *tiles, const uint8_t *scales, uint32_t m, uint32_t n,
                                const uint16_t *x, uint32_t x_stride, uint32_t rows, unsigned long long *partials,
                                uint32_t *out, uint32_t n_cus, bool f16, KernelTimer *timer, float softcap, float *out_conf) {
    const dim3 grid(greedy_segments(m, n_cus));
    float2 *conf_part = reinterpret_cast<float2 *>(partials + (size_t)FFMOE_MAX_VERIFY_ROWS * grid.x);
#define FFMOE_GREEDY(H, C)                                                                                                  \
    hipLaunchKernelGGL((once ? matrix_gemv_kernel<true, H, true, C, false, 0, false, true> : matrix_gemv_kernel<true, H, true, C>), grid, dim3(256), 0, s, \
                       tiles, scales, m, n / kGroup, x, x_stride, rows, partials, 0u, conf_part, softcap)
    // (16 rows, N = 2,112, us without the hint | with: 259 MB 62.7 | 62.8, 270 MB 69.6 | 70.4, 301 MB 76.2 | 75.4, 338 MB 84.8 | 82.8)
    const bool once = (size_t)((m + 31) / 32) * (n / kGroup) * kTileBytes > kMemoryCacheBytes;
    if (f16) { if (out_conf) FFMOE_GREEDY(true, true); else FFMOE_GREEDY(true, false); }
    else { if (out_conf) FFMOE_GREEDY(false, true); else FFMOE_GREEDY(false, false); }
#undef FFMOE_GREEDY
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    timer->mark(s, FFMOE_K_GEMV);
    hipLaunchKernelGGL(argmax_final_kernel, dim3(rows), dim3(256), 0, s, partials, grid.x, out, conf_part, softcap, out_conf);
    timer->mark(s, FFMOE_K_ARGMAX);
    return hipGetLastError();
}

bool argmax_takes_scratch(uint32_t rows, uint32_t count) {
    return count > kArgmaxOneBlock && rows <= FFMOE_MAX_VERIFY_ROWS && count <= kSampleMaxSegments * kSampleSegment;
}

hipError_t launch_argmax_rows(hipStream_t s, const float *logits, uint32_t stride, uint32_t rows, uint32_t count, float softcap,
                              uint32_t *out, float *out_conf, SampleScratch sc) {
    if (sc.segments && argmax_takes_scratch(rows, count)) {
        const uint32_t n_seg = (count + kSampleSegment - 1) / kSampleSegment;
        hipLaunchKernelGGL(argmax_rows_kernel<256>, dim3(rows, n_seg), dim3(256), 0, s, logits, stride, count, kSampleSegment, softcap, out,
                           out_conf, sc.segments);
        hipLaunchKernelGGL(argmax_merge_kernel, dim3(rows), dim3(256), 0, s, sc.segments, n_seg, softcap, out, out_conf);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(argmax_rows_kernel<kArgmaxThreads>, dim3(rows), dim3(kArgmaxThreads), 0, s, logits, stride, count, count, softcap, out,
                       out_conf, (SampleSegment *)nullptr);
    return hipGetLastError();
}

}  // namespace ffmoe
