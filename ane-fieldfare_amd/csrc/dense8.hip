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

constexpr int kTilesN = 8;                                  // 16-row tiles per 128-row block
constexpr int kBFrags = kTilesN * 2;                        // weight fragments of it per group

__device__ __forceinline__ uint32_t ext_groups(uint32_t n_groups) { return (3 * n_groups + kGroup - 1) / kGroup; }

// Column c of the bias columns, row j of a 16-row block: where it stands behind the block's (or tile's) groups.
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
        const bool real = tr < n_tiles;                     // tiles past the matrix (half a block): zeros
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

// The GEMMs. An item = 16 NM rows x one N-block of 256 weight rows, a block of eight waves: wave w has the two 16-row tiles 2 w and
// 2 w + 1 (GATED: gate and up of the same 16 activations) for all the rows. Inputs and weights lie in operand order and go straight
// into LDS, a fragment (1 KiB) per instruction, two groups ahead: the inputs into a ring of three groups that the block shares,
// a wave's 4 KiB of weights into two slots of its own, from where they go to registers. One barrier per group; it stands where the
// last of a group's fragments have been read, so that reads run on into the next group and the buffer can be filled again.
// Two fma per product bring a group's sums into the running ones with their scale: those of a 16-row block stand between the
// products of the next (a group's last block: of the next group's first). GATED: out = the activations as the second GEMM's
// operands (with their group sums); else out = the output rows.
// Bound: the matrix unit and, with it on all compute units, the card's power: the products, their fma and the fragment reads
// alone take 53 us where the gated product of 13 blocks takes 65 on 68 compute units and 80 on 255 (with inputs of zeros 72). The
// barrier and the weights' reads are 6 of the difference, the loads into LDS 8; nearer loads change nothing, nor do four products
// in a row with a raised wave priority, weights in two register sets without moves, or offsets in vector registers. 2,816 ->
// 2,112 -> 2,816, us of gate/up + down where four waves took 64 or 128 rows and 128 weight rows with weights through registers and
// a barrier before every group's reads | now: 640 rows 42 + 27 | 30 + 21, 1,024 rows 55 + 32 | 38 + 23, 3,072 rows 115 + 61 | 80 +
// 46, 8,192 rows 261 + 130 | 230 + 118; FP16 alike. 704 -> 2,816, 1,024 rows 21 + 31 | 17 + 25; 2,816 -> 256, 4,096 rows 45 + 16 |
// 28 + 15.

// LDS of a block: three groups of inputs (2 NM KiB each), then every wave's two groups of weights and of their scales. The
// epilogue's images take the same bytes.
constexpr int kWaves8 = 8;
constexpr uint32_t kFrag8 = kWave * 16;                     // bytes of a fragment
constexpr uint32_t kSlot8 = 4 * kFrag8, kScaleSlot8 = kWave * 4;
template <int NM> struct Lds8 {
    static constexpr uint32_t a_bytes = 2 * NM * kFrag8, w_at = 3 * a_bytes, s_at = w_at + 2 * kWaves8 * kSlot8,
                              bytes = s_at + 2 * kWaves8 * kScaleSlot8;
};
constexpr int kMaxBlocks8 = 15, kMinBlocks8 = 3;            // 16-row blocks per item

// Fragments of inputs in flight or in use per wave: a divisor of a group's 2 NM, so that a fragment's registers are known at compile time.
constexpr int queue8(int nm) {
    int q = 2;
    for (int d = 3; d <= (nm == 11 || nm == 13 ? nm : 8); ++d)
        if (2 * nm % d == 0) q = d;
    return q;
}

template <bool GATED, int NM, bool F16>
__global__ __launch_bounds__(64 * kWaves8, 2) void dense8_gemm_kernel(const uint8_t *__restrict__ weights, const float *__restrict__ scales,
                                                                      uint32_t n_groups, uint32_t n_blocks, uint32_t n_cols,
                                                                      const uint8_t *__restrict__ a, uint32_t t, uint16_t *__restrict__ out,
                                                                      uint32_t out_stride) {
    using L = Lds8<NM>;
    __shared__ __align__(16) uint8_t lds[L::bytes];
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), j = lane & 15, jq = lane >> 4;
    // the items N-block by N-block, an eighth of the list per XCD: each reads its eighth of the weights into its L2 once
    const uint32_t row_blocks = (t + 15) / 16, m_tiles = (row_blocks + NM - 1) / NM, n_nb = (n_blocks + 1) / 2, all = m_tiles * n_nb;
    const uint32_t xcd = blockIdx.x & 7, first = (uint32_t)((uint64_t)all * xcd / 8);
    const uint32_t item = first + (blockIdx.x >> 3);
    if (item >= (uint32_t)((uint64_t)all * (xcd + 1) / 8)) return;
    const uint32_t nb = item / m_tiles, block0 = item % m_tiles * NM;
    const uint32_t all_groups = n_groups + ext_groups(n_groups), last = all_groups - 1;
    // this wave's 128-row block of weights, of which it has tiles 2 (wave % 4) and the next; past the last block the last again
    const bool owns = nb * 2 + (wave >> 2) < n_blocks;
    const size_t wblock = (size_t)min(nb * 2 + (wave >> 2), n_blocks - 1) * all_groups;
    const uint8_t *const w = weights + (wblock * kBFrags + (wave & 3) * 4) * kFrag8;
    const float *const sc_src = scales + wblock * (16 * kTilesN) + (wave & 3) * 2;
    const uint32_t sc_lane = ((lane & 31) >> 1) * (kTilesN * 4) + (lane & 1) * 4;        // row by row, both tiles
    constexpr int kLoadsA = (2 * NM + kWaves8 - 1) / kWaves8;                              // KiB per wave and group
    constexpr int kLoads = kLoadsA + 5;
    uint32_t from[kLoadsA], to[kLoadsA];
#pragma unroll
    for (int k = 0; k < kLoadsA; ++k) {
        // (what does not divide by the waves, the last fragment several times; blocks past the last are the last again, never stored)
        const uint32_t piece = min(wave + kWaves8 * k, 2u * NM - 1);
        from[k] = min(block0 + (piece >> 1), row_blocks - 1) * all_groups * 2 + (piece & 1);
        to[k] = piece * kFrag8;
    }
    auto load_w = [&](uint32_t grp, uint32_t slot, int k) __attribute__((always_inline)) {
        if (k < 4) global_to_lds_16(w + (size_t)grp * (kBFrags * kFrag8) + k * kFrag8, lane * 16, lds_base + L::w_at + (slot * kWaves8 + wave) * kSlot8 + k * kFrag8);
        else global_to_lds_4(sc_src + grp * (16 * kTilesN), sc_lane, lds_base + L::s_at + (slot * kWaves8 + wave) * kScaleSlot8);
    };
    auto load_a = [&](uint32_t grp, uint32_t buf, int k) __attribute__((always_inline)) {
        global_to_lds_16(a + ((size_t)from[k] + 2 * grp) * kFrag8, lane * 16, lds_base + buf + to[k]);
    };
    uint4 wf[2][2];                     // operands: tile, k-half
    float sc[2][2] = {};                // of the group before, of this one
    uint4 wn[2][2];
    float sn[2];
    auto read_w = [&](uint32_t slot) __attribute__((always_inline)) {
        const uint8_t *at = lds + L::w_at + (slot * kWaves8 + wave) * kSlot8;
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int kh = 0; kh < 2; ++kh) wn[st][kh] = *reinterpret_cast<const uint4 *>(at + (st * 2 + kh) * kFrag8 + lane * 16);
        const float2 v = *reinterpret_cast<const float2 *>(lds + L::s_at + (slot * kWaves8 + wave) * kScaleSlot8 + j * 8);
        sn[0] = v.x, sn[1] = v.y;
    };
    constexpr int kFrags = 2 * NM, kQueue = queue8(NM), kLate = 2;
    uint4 xq[kQueue];
    auto read_a = [&](uint32_t buf, int f) __attribute__((always_inline)) {
        xq[f % kQueue] = *reinterpret_cast<const uint4 *>(lds + buf + f * kFrag8 + lane * 16);
    };
    f32x4 tot[NM][2];
#pragma unroll
    for (int i = 0; i < NM; ++i) tot[i][0] = tot[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    // a block's products of one group, in flight while the block before is added up (a group's last during the next one's first)
    f32x4 part[3][2];
    part[2][0] = part[2][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto part_of = [](int i) __attribute__((always_inline)) { return i == NM - 1 ? 2 : i & 1; };
    auto add = [&](int i, int m, int which) __attribute__((always_inline)) {              // two of a block's eight sums
        const int st = m >> 1;
#pragma unroll
        for (int r = 2 * (m & 1); r < 2 * (m & 1) + 2; ++r) tot[i][st][r] = __builtin_fmaf(sc[st][which], part[part_of(i)][st][r], tot[i][st][r]);
    };
    uint32_t cur = 0, next = L::a_bytes, before = 2 * L::a_bytes, slot = 0;

    // H: the element type of this group's operands (the bias columns are bf16 in either mode)
    auto step = [&](uint32_t grp, auto type) __attribute__((always_inline)) {
        constexpr bool H = decltype(type)::value;
#pragma unroll
        for (int st = 0; st < 2; ++st) wf[st][0] = wn[st][0], wf[st][1] = wn[st][1], sc[st][0] = sc[st][1], sc[st][1] = sn[st];
        constexpr int kBarrier = kFrags - kQueue + 1 + kLate;
#pragma unroll
        for (int f = 0; f < kFrags; ++f) {
            const int i = f >> 1, kh = f & 1, ahead = f + kQueue - 1;
            if (f == kBarrier) {
                ring_barrier<kLoads>();
                read_w(slot ^ 1);
#pragma unroll
                for (int n = 0; n < kLate; ++n) read_a(next, n);
            }
            if (ahead < kFrags) read_a(cur, ahead);
            else if (f >= kBarrier) read_a(next, ahead - kFrags);
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
                part[part_of(i)][st] = Act<H>::mfma(xq[f % kQueue], wf[st][kh], kh ? part[part_of(i)][st] : zero);
                // the sums of the block before, three products behind their last one
                const int at = 2 * f + st, m = at & 3;
                if (m > 0) add((i + NM - 1) % NM, m - 1, i > 0);
                else if (at > 0) add((i + NM - 2) % NM, 3, i > 1);
#pragma unroll
                for (int k = 0; k < 5; ++k)
                    if (at == 2 + k * (2 * kBarrier - 2) / 5) load_w(min(grp + 2, last), slot, k);
#pragma unroll
                for (int k = 0; k < kLoadsA; ++k)
                    if (at == 2 * kBarrier + 1 + k * (2 * (kFrags - kBarrier) - 1) / kLoadsA) load_a(min(grp + 3, last), cur, k);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        add((2 * NM - 2) % NM, 3, 1);
        const uint32_t c = cur;
        cur = next, next = before, before = c;
        slot ^= 1;
    };
#pragma unroll
    for (uint32_t g = 0; g < 3; ++g) {
#pragma unroll
        for (int k = 0; k < kLoadsA; ++k) load_a(min(g, last), g * L::a_bytes, k);
#pragma unroll
        for (int k = 0; k < 5; ++k)
            if (g < 2) load_w(min(g, last), g, k);
    }
    vmem_barrier<kLoads + kLoadsA>();
    read_w(0);
#pragma unroll
    for (int f = 0; f < kQueue - 1; ++f) read_a(cur, f);
#pragma nounroll
    for (uint32_t grp = 0; grp < n_groups; ++grp) step(grp, std::integral_constant<bool, F16>{});
#pragma nounroll
    for (uint32_t grp = n_groups; grp < all_groups; ++grp) step(grp, std::integral_constant<bool, false>{});
#pragma unroll
    for (int m = 0; m < 4; ++m) add(NM - 1, m, 1);
    // (an fp32 value like the others' and then a 16-bit one: not both in one instruction with one rounding)
    asm volatile("" : "+v"(tot[NM - 1][0]), "+v"(tot[NM - 1][1]));
    vmem_barrier<0>();                                      // no load is on its way into what the epilogue writes
    lds_barrier();

    // lane (j, jq) holds weight row j of both tiles for rows 4 jq .. 4 jq + 3 of every 16-row block
    if constexpr (GATED) {
        // gate and up of 16 activations: a quarter of group 2 nb + wave / 4 of F, k-half (wave / 2) % 2. The operands are put together
        // in LDS ([group][16-row block][k-half][lane]), stored from there, and their groups summed there.
        uint16_t *img = reinterpret_cast<uint16_t *>(lds);
#pragma unroll
        for (int i = 0; i < NM; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float g = Act<F16>::widen(Act<F16>::round(tot[i][0][r])), u = Act<F16>::widen(Act<F16>::round(tot[i][1][r]));
                img[((((wave >> 2) * NM + i) * 2 + (wave >> 1 & 1)) * kWave + ((wave & 1) * 2 + (j >> 3)) * 16 + 4 * jq + r) * 8 + (j & 7)] =
                    Act<F16>::round(gelu_tanh_fast(g) * u);
            }
        lds_barrier();
        const uint32_t f_groups = n_blocks, f_all = f_groups + ext_groups(f_groups), groups = min(2u, f_groups - 2 * nb);
        for (uint32_t p = tid; p < groups * NM * 2 * kWave; p += 64 * kWaves8) {
            const uint32_t gi = p / (NM * 2 * kWave), i = p / (2 * kWave) % NM;
            if (block0 + i < row_blocks)
                reinterpret_cast<uint4 *>(out)[((size_t)(block0 + i) * f_all + 2 * nb + gi) * (2 * kWave) + p % (2 * kWave)] = reinterpret_cast<const uint4 *>(lds)[p];
        }
        // the group sums of the activations as they were rounded, into the second GEMM's bias columns: a thread per row and group
        for (uint32_t p = tid; p < groups * NM * 16; p += 64 * kWaves8) {
            const uint32_t gi = p / (NM * 16), i = p / 16 % NM, row = p & 15;
            if (block0 + i >= row_blocks) continue;
            float sum[2];
#pragma unroll
            for (int kh = 0; kh < 2; ++kh) {
                const uint4 *at = reinterpret_cast<const uint4 *>(lds) + ((gi * NM + i) * 2 + kh) * kWave + row;
                float v[16];
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const uint4 x = at[16 * c], y = at[16 * (c + 2)];
                    const uint32_t xw[4] = {x.x, x.y, x.z, x.w}, yw[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        v[8 * c + 2 * q] = Act<F16>::lo(xw[q]) + Act<F16>::lo(yw[q]);
                        v[8 * c + 2 * q + 1] = Act<F16>::hi(xw[q]) + Act<F16>::hi(yw[q]);
                    }
                }
#pragma unroll
                for (int m = 1; m < 16; m <<= 1)
#pragma unroll
                    for (int q = 0; q < 16; q += 2 * m) v[q] += v[q + m];
                sum[kh] = v[0];
            }
            uint16_t part[3];
            split_sum(sum[0] + sum[1], part);
            uint16_t *dst = out + (size_t)(block0 + i) * f_all * 2 * (kWave * 8);
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const uint32_t c = 3 * (2 * nb + gi) + q;
                dst[((size_t)(f_groups + (c >> 6)) * 2 + ((c & 63) >> 5)) * (kWave * 8) + ext_lane(c, row) * 8 + (c & 7)] = part[q];
            }
        }
    } else {
        // a 16-row block of this wave's columns is 16 rows x 64 bytes: each wave turns its blocks through a piece of LDS of its own
        constexpr uint32_t kStageRow = 64 + 16, kStage = 16 * kStageRow;                 // bytes: 32 columns + padding
        constexpr int kTurn = 4;
        static_assert(kWaves8 * kTurn * kStage <= L::bytes, "staging fits the rings");
        uint8_t *stage = lds + wave * (kTurn * kStage);
        const uint32_t sub = lane >> 2, chunk = lane & 3, col = nb * 256 + wave * 32 + 8 * chunk;
        if (!owns) return;
#pragma unroll
        for (int i0 = 0; i0 < NM; i0 += kTurn) {
#pragma unroll
            for (int i = i0; i < i0 + kTurn && i < NM; ++i)
#pragma unroll
                for (int st = 0; st < 2; ++st)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        *reinterpret_cast<uint16_t *>(stage + (i - i0) * kStage + (4 * jq + r) * kStageRow + st * 32 + 2 * j) = Act<F16>::round(tot[i][st][r]);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
            for (int i = i0; i < i0 + kTurn && i < NM; ++i) {
                const uint32_t row = (block0 + i) * 16 + sub;
                const uint4 v = *reinterpret_cast<const uint4 *>(stage + (i - i0) * kStage + sub * kStageRow + 16 * chunk);
                if (row < t && col < n_cols) *reinterpret_cast<uint4 *>(out + (size_t)row * out_stride + col) = v;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }
}

uint32_t all_groups_of(uint32_t n) { return n / kGroup + (3 * (n / kGroup) + kGroup - 1) / kGroup; }
// 16-row blocks per item: as many as make the rounds of items over the compute units cheapest, an item of n costing n + 6 (2,816 wide,
// one round: 28.7 us at 3, 68.2 at 15). Of 3..15 each, the rule's is the fastest or within 4% of it, gate/up of 2,112 at 640 rows
// (3: 29 us, 8: 45), 1,024 (5: 36, 4: 61 in two rounds), 2,048 (9: 56, 8: 92), 3,072 (13: 80, 12: 125, 7: 90), 4,096 (9: 108, 12:
// 122), 8,192 (12: 203, 9: 214, 13: 222); down at 3,072 (9: 44, 8: 70, 13: 54), 4,096 (12: 54, 11: 89). 15 is what LDS holds; below 3
// a group's 32 KiB of weights take longer than its products. Any gives the same bits.
uint32_t dense8_blocks(uint32_t row_blocks, uint32_t n_nb, uint32_t n_cus) {
    uint32_t best = kMaxBlocks8;
    uint64_t least = ~0ull;
    for (uint32_t n = kMaxBlocks8; n >= (uint32_t)kMinBlocks8; --n) {
        const uint64_t rounds = ((row_blocks + n - 1) / n * n_nb + n_cus - 1) / n_cus, cost = rounds * (6 + n);
        if (cost < least) least = cost, best = n;
    }
    return best;
}
uint32_t n_blocks_of(uint32_t stored_rows) { return (stored_rows / 16 + kTilesN - 1) / kTilesN; }

}  // namespace

// While its items are fewer than the compute units, a GEMM here takes one item's chain of groups however few the rows, where the
// library's two take 22 us and 12.5 us per 1,000 rows and 10^6 weights of a projection: the lines cross where rows * d f / 10^6 is 68
// times the groups of both products less 2,000 (fitted at 18 widths, GPU time, when a group of the chain took 0.7 us). A group is
// 0.5 us now and the forms cross lower: library form | this one, us: 2,816 -> 2,112, 704 rows 76 | 56, 3,072 rows 248 | 140; 2,816 ->
// 704, 1,024 rows 55 | 45; 1,024 -> 2,816, 1,024 rows 67 | 50. The line of narrow layers stays: a chunk keeps the form, and with it the
// bits, that it had. Wide ones change at 385 rows, where the library's form takes a step up: 2,816 -> 2,112, 301 rows 47 | 48, 384 rows 50 | 49,
// 400 rows 65 | 49, 448 rows 68 | 50, 639 rows 63 | 50; 2,816 -> 1,600, 385 rows 50 | 45, 512 rows 53 | 46; 2,304 -> 1,792 46 | 42, 51 | 42; 2,048 -> 2,048 46 | 41, 49 | 42 (FP16 alike; errors against 64 bits equal: 3.32e-3, FP16 4.16e-4), those from
// 2.8 * 10^6 weights of a projection at 560: 2,816 -> 1,024, 448 rows 40 | 41, 560 rows 45 | 42; 1,728 -> 1,664, 400 rows 37 | 38, 560 rows 44 | 38.
// Narrower, 2,816 -> 704, 560 rows 38 | 40. Else not below 640 rows, where the forms met at the widest, nor beyond 1,024, where the narrowest (2,816 -> 256) still
// crossed, but in a call that the library's own 41 us on the host bound.
uint32_t dense8_min_rows(uint32_t d, uint32_t f) {
    if ((uint64_t)d * f >= 2800000) return (uint64_t)d * f >= 4000000 ? 385 : 560;
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
    const uint32_t nm = dense8_blocks(row_blocks, (n_blocks + 1) / 2, n_cus), all = (row_blocks + nm - 1) / nm * ((n_blocks + 1) / 2);
    const dim3 grid((all + 7) / 8 * 8);
    auto launch = [&](auto blocks) {
        constexpr int N = decltype(blocks)::value;
        hipLaunchKernelGGL((gated ? (f16 ? dense8_gemm_kernel<true, N, true> : dense8_gemm_kernel<true, N, false>)
                                  : (f16 ? dense8_gemm_kernel<false, N, true> : dense8_gemm_kernel<false, N, false>)),
                           grid, dim3(64 * kWaves8), 0, s, static_cast<const uint8_t *>(weights), scales, n / kGroup, n_blocks, stored_rows,
                           static_cast<const uint8_t *>(ops), t, static_cast<uint16_t *>(out), out_stride);
    };
#define FFMOE_DENSE8(N) case N: launch(std::integral_constant<int, N>{}); break
    switch (nm) {
        FFMOE_DENSE8(3);
        FFMOE_DENSE8(4);
        FFMOE_DENSE8(5);
        FFMOE_DENSE8(6);
        FFMOE_DENSE8(7);
        FFMOE_DENSE8(8);
        FFMOE_DENSE8(9);
        FFMOE_DENSE8(10);
        FFMOE_DENSE8(11);
        FFMOE_DENSE8(12);
        FFMOE_DENSE8(13);
        FFMOE_DENSE8(14);
        default: launch(std::integral_constant<int, 15>{}); break;
    }
#undef FFMOE_DENSE8
    return hipGetLastError();
}

}  // namespace ffmoe
