// The sampled choice over rows of fp32 logits (sample_rows_f32, Metal/Sampling/logit.metal:1010-1259; dispatched by
// LMHeadChainInt4.encodeChoice, Kernels/Fusions/LMHeadChainInt4.swift:192-223): per row one draw from the tempered
// softmax of the soft-capped logits by the Gumbel-max rule,
//     token = argmax_i  capped(logit_i) / T + G(seed, key, token_i),
// over the entries the truncation keeps. The noise is a counter-based hash of (seed, position key, token id), so every
// producer that draws a position draws the same noise. Truncation in the sampler's order: the top_k largest capped
// logits (ties to the lower index), of those the shortest prefix whose T = 1 probability mass reaches top_p, then
// the draw at temperature T over the survivors.
//
// Two forms with the same survivors. Long rows (use_scan below) take two launches: blocks of 2,048 logits sweep the row
// ONCE - one wave per 64 logits leaves their largest capped value, a block its share of the normaliser (or, without
// truncation, its own winner of the draw) - and one block per row finishes from those: the want-th largest of the 64-wide
// groups' maxima is a lower bound of the want-th largest logit, only groups that reach it can hold a survivor, and
// what those hold above the bound (a few hundred logits) is ranked exactly. One row of 262,144 logits, top_k = 64: 375 us as
// one block's five sweeps (tanhf per logit and sweep, and LDS histograms whose few occupied bins serialise the
// atomics) -> 17 us; sixteen rows without truncation 20 us.
// Short rows, and rows whose groups tie at the bound in numbers that overflow the candidate lists, take one block of
// 1,024 threads per row. Without truncation: two sweeps (the largest capped logit; the draw and the normaliser). With it
// the k-th largest is found EXACTLY by a radix select over the order-preserving integer image of the capped logits -
// three sweeps with LDS histograms of 11, 11 and 10 bits; a fourth sweep gathers the values above the threshold (any
// order: they are ranked afterwards) and, of the values equal to it, the lowest indices (in index order, wave by wave).
// The <= 256 candidates are ranked by counting, thread 0 walks the top_p prefix, and the survivors draw.
#include <hip/hip_runtime.h>

#include <cfloat>

#include "common.hpp"
#include "kernels.hpp"
#include "topk.hpp"

namespace ffmoe {
namespace {

constexpr int kSampleThreads = 1024, kSampleWaves = kSampleThreads / 64;
constexpr int kSampleMaxK = 256;

struct SampleRule {
    float temperature, top_p;
    uint32_t top_k, key_base;
    float softcap;
    uint32_t seed_lo, seed_hi;
};

// logits are capped to (-cap, cap); a non-finite logit never takes part (logit.metal:1055-1057)
__device__ __forceinline__ float sample_capped(float v, float cap) {
    return (v - v == 0.0f) ? cap * tanhf(v / cap) : -INFINITY;
}

// Standard Gumbel noise from the hash of (seed, key, token): one SplitMix64 step of the mixed state, its top 24 bits
// as a uniform in (0, 1) (logit.metal:1042-1051).
__device__ __forceinline__ float sample_gumbel(unsigned long long seed, uint32_t key, uint32_t token) {
    unsigned long long z = seed ^ ((unsigned long long)key * 0x9E3779B97F4A7C15ull) ^ ((unsigned long long)token * 0xD1B54A32D192ED03ull);
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    const float u = ((float)(uint32_t)(z >> 40) + 0.5f) * (1.0f / 16777216.0f);
    return -logf(-logf(u));
}

// float -> unsigned, order preserving (-inf lowest of the values that occur here)
__device__ __forceinline__ uint32_t sample_key(float v) {
    const uint32_t b = __float_as_uint(v);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

struct SampleShared {
    uint32_t hist[2048];
    float red_f[kSampleWaves];
    unsigned long long red_k[kSampleWaves];
    uint32_t wave_eq[kSampleWaves][kSampleMaxK];     // per wave: the first indices (in index order) whose value equals the threshold
    uint32_t wave_eq_n[kSampleWaves];
    float cand_v[kSampleMaxK], sorted_v[kSampleMaxK];
    uint32_t cand_i[kSampleMaxK], sorted_i[kSampleMaxK];
    uint32_t n_above, bin, above;
};

// How many lanes below this one have their bit set.
__device__ __forceinline__ uint32_t lanes_in_front(unsigned long long mask) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// Lane l: the sum over lanes 0 .. l (register moves; a shift by __shfl_up is a trip through LDS at each of the six steps).
__device__ __forceinline__ float wave_running_sum(float v) {
    auto from = [](float x, auto ctrl, auto rows) {
        return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), decltype(ctrl)::value, decltype(rows)::value, 0xF, false));
    };
    using std::integral_constant;
    v += from(v, integral_constant<int, 0x111>{}, integral_constant<int, 0xF>{});   // row_shr:1, 2, 4, 8: sums inside a row of 16
    v += from(v, integral_constant<int, 0x112>{}, integral_constant<int, 0xF>{});
    v += from(v, integral_constant<int, 0x114>{}, integral_constant<int, 0xF>{});
    v += from(v, integral_constant<int, 0x118>{}, integral_constant<int, 0xF>{});
    v += from(v, integral_constant<int, 0x142>{}, integral_constant<int, 0xA>{});   // row_bcast:15 into rows 1 and 3
    v += from(v, integral_constant<int, 0x143>{}, integral_constant<int, 0xC>{});   // row_bcast:31 into rows 2 and 3
    return v;
}

__device__ __forceinline__ float block_max_f(float v, SampleShared &sh) {
    v = wave_max_f32(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh.red_f[threadIdx.x >> 6] = v;
    __syncthreads();
    float r = sh.red_f[0];
    for (int w = 1; w < kSampleWaves; ++w) r = fmaxf(r, sh.red_f[w]);
    return r;
}

// sum in a fixed order: lanes by xor-butterfly, then the waves one after the other
__device__ __forceinline__ float block_sum_f(float v, SampleShared &sh) {
    v = wave_butterfly_sum(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh.red_f[threadIdx.x >> 6] = v;
    __syncthreads();
    float r = 0.0f;
    for (int w = 0; w < kSampleWaves; ++w) r += sh.red_f[w];
    return r;
}

// two sums side by side
__device__ __forceinline__ float2 block_sum_f2(float2 v, SampleShared &sh) {
    v = make_float2(wave_butterfly_sum(v.x), wave_butterfly_sum(v.y));
    float2 *red = reinterpret_cast<float2 *>(sh.red_k);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float2 r = make_float2(0.0f, 0.0f);
    for (int w = 0; w < kSampleWaves; ++w) {
        r.x += red[w].x;
        r.y += red[w].y;
    }
    return r;
}

__device__ __forceinline__ unsigned long long block_max_k(unsigned long long v, SampleShared &sh) {
    v = wave_max_key(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh.red_k[threadIdx.x >> 6] = v;
    __syncthreads();
    unsigned long long r = sh.red_k[0];
    for (int w = 1; w < kSampleWaves; ++w) r = sh.red_k[w] > r ? sh.red_k[w] : r;
    return r;
}

// Of `bins` histogram counts (a multiple of 64, <= 2048) find, from the top, the bin that holds the want-th largest
// entry (1-based): sh.bin = that bin, sh.above = entries in the bins above it. Run by the whole block (wave 0 works).
__device__ __forceinline__ void find_bin(SampleShared &sh, uint32_t bins, uint32_t want) {
    __syncthreads();
    if (threadIdx.x < 64) {
        const uint32_t lane = threadIdx.x, per = bins / 64;
        // lane l owns the bins [bins - per (l + 1), bins - per l): lane 0 the highest
        const uint32_t hi = bins - per * lane;
        uint32_t mine = 0;
        for (uint32_t b = 0; b < per; ++b) mine += sh.hist[hi - 1 - b];
        uint32_t incl = mine;                      // entries in this lane's bins and all higher lanes'
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t up = (uint32_t)__shfl_up((int)incl, o, 64);
            if (lane >= (uint32_t)o) incl += up;
        }
        const uint32_t before = incl - mine;
        if (before < want && want <= incl) {
            uint32_t acc = before;
            for (uint32_t b = 0; b < per; ++b) {
                const uint32_t c = sh.hist[hi - 1 - b];
                if (acc + c >= want) {
                    sh.bin = hi - 1 - b;
                    sh.above = acc;
                    break;
                }
                acc += c;
            }
        }
    }
    __syncthreads();
}

// The end of a truncated draw, called by the whole block: sh.sorted_v / sorted_i hold the n largest in order. The top_p prefix
// over the T = 1 distribution within the top k (logit.metal:1213-1224; `total1` = the normaliser over the whole row), then
// the draw at temperature T over the survivors. Wave 0 does it alone, four ranks per lane: no barrier in the chain.
__device__ __forceinline__ void sample_finish(SampleShared &sh, const SampleRule &p, uint32_t n, float total1, unsigned long long seed,
                                              uint32_t key, const uint32_t *__restrict__ ids, uint32_t *__restrict__ out_token,
                                              float *__restrict__ out_prob) {
    constexpr int kSlots = kSampleMaxK / 64;
    const float invT = 1.0f / p.temperature;
    __syncthreads();
    if (threadIdx.x >= 64) return;
    const uint32_t lane = threadIdx.x;
    float v[kSlots];                                            // lane l, slot u: rank 64 u + l
    uint32_t at[kSlots];
#pragma unroll
    for (int u = 0; u < kSlots; ++u) {
        const uint32_t rank = min(64u * u + lane, n - 1);
        v[u] = sh.sorted_v[rank];
        at[u] = sh.sorted_i[rank];
    }
    const float top = __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(v[0])));
    float share[kSlots], incl[kSlots], score[kSlots];
    float so_far = 0.0f;
    // (also of those that the prefix leaves out: beside its chain instead of behind it)
#pragma unroll
    for (int u = 0; u < kSlots; ++u) {
        if (64u * u >= n) break;
        score[u] = v[u] * invT + sample_gumbel(seed, key, ids ? ids[at[u]] : at[u]);
    }
#pragma unroll
    for (int u = 0; u < kSlots; ++u) {
        share[u] = 64u * u + lane < n ? expf(v[u] - p.softcap) / total1 : 0.0f;
        incl[u] = share[u];
    }
#pragma unroll
    for (int u = 0; u < kSlots; ++u) {
        if (64u * u >= n) break;
        incl[u] = wave_running_sum(incl[u]) + so_far;
        so_far = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(incl[u]), 63));
    }
    // The prefix is defined by the running sum that takes the shares one after the other. Two orders of adding <= 256
    // positive shares that add to at most about 1 differ by less than 256 * 2^-24 * 2: where no prefix sum comes closer to
    // top_p than that, the scan decides; else (equal logits whose shares meet top_p exactly) the sum itself runs.
    constexpr float kClose = 4e-5f;
    uint32_t keep = n;
    bool close = false;
#pragma unroll
    for (int u = kSlots - 1; u >= 0; --u) {
        if (64u * u >= n) continue;
        const bool in = 64u * u + lane < n;
        const unsigned long long over = __ballot(in && incl[u] >= p.top_p);
        close = close || __ballot(in && fabsf(incl[u] - p.top_p) < kClose) != 0ull;
        if (over) keep = 64u * u + (uint32_t)__builtin_ctzll(over) + 1;
    }
    if (close) {
        keep = n;
        float cum = 0.0f;
#pragma unroll
        for (int u = 0; u < kSlots; ++u)
            for (uint32_t l = 0; l < 64 && 64u * u + l < n && keep == n; ++l) {
                cum += __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(share[u]), (int)l));
                if (cum >= p.top_p) keep = min(n, 64u * u + l + 1);
            }
    }
    unsigned long long best = 0ull;
    float esum = 0.0f;
#pragma unroll
    for (int u = 0; u < kSlots; ++u) {
        if (64u * u >= keep) break;
        const uint32_t rank = 64u * u + lane;
        float e = 0.0f;
        unsigned long long mine = 0ull;
        if (rank < keep) {
            e = expf((v[u] - top) * invT);
            mine = ((unsigned long long)sample_key(score[u]) << 32) | (0xFFFFFFFFu - rank);
        }
        mine = wave_max_key(mine);
        esum += wave_butterfly_sum(e);
        best = mine > best ? mine : best;
    }
    if (lane == 0) {
        const uint32_t bj = 0xFFFFFFFFu - (uint32_t)best;
        *out_token = sh.sorted_i[bj];
        *out_prob = expf((sh.sorted_v[bj] - top) * invT) / esum;
    }
}

// One row by one block of kSampleThreads threads, whatever it holds.
__device__ void sample_one_row(SampleShared &sh, const float *__restrict__ row, uint32_t count, const uint32_t *__restrict__ ids,
                               const SampleRule &p, uint32_t key, uint32_t *__restrict__ out_token, float *__restrict__ out_prob) {
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const float cap = p.softcap, invT = 1.0f / p.temperature;
    const unsigned long long seed = ((unsigned long long)p.seed_hi << 32) | p.seed_lo;
    const bool truncated = p.top_k > 0u && p.top_k < count;
    auto token_of = [&](uint32_t i) { return ids ? ids[i] : i; };

    if (!truncated) {
        float m = -INFINITY;
        for (uint32_t i = tid; i < count; i += kSampleThreads) m = fmaxf(m, sample_capped(row[i], cap));
        m = block_max_f(m, sh);
        unsigned long long best = 0ull;
        float sum = 0.0f;
        for (uint32_t i = tid; i < count; i += kSampleThreads) {
            const float c = sample_capped(row[i], cap);
            if (c == -INFINITY) continue;
            sum += expf((c - m) * invT);
            const float g = c * invT + sample_gumbel(seed, key, token_of(i));
            const unsigned long long k = ((unsigned long long)sample_key(g) << 32) | (0xFFFFFFFFu - i);
            best = k > best ? k : best;
        }
        best = block_max_k(best, sh);
        const float total = block_sum_f(sum, sh);
        if (tid == 0) {
            const uint32_t j = best ? 0xFFFFFFFFu - (uint32_t)best : 0xFFFFFFFFu;
            *out_token = j;
            *out_prob = (j == 0xFFFFFFFFu || !(total > 0.0f)) ? 0.0f : expf((sample_capped(row[j], cap) - m) * invT) / total;
        }
        return;
    }

    // ---- exact top_k: radix select on the keys of the capped logits, 11 + 11 + 10 bits -------------------------
    const uint32_t k = p.top_k;
    float s1 = 0.0f;
    for (uint32_t b = tid; b < 2048; b += kSampleThreads) sh.hist[b] = 0;
    if (tid < kSampleWaves) sh.wave_eq_n[tid] = 0;
    if (tid == 0) sh.n_above = 0;
    __syncthreads();
    uint32_t n_finite = 0;
    for (uint32_t i = tid; i < count; i += kSampleThreads) {
        const float c = sample_capped(row[i], cap);
        if (c == -INFINITY) continue;
        s1 += expf(c - cap);                                   // the T = 1 normaliser, offset by the cap
        ++n_finite;
        atomicAdd(&sh.hist[sample_key(c) >> 21], 1u);
    }
    const float total1 = block_sum_f(s1, sh);
    const uint32_t finite = (uint32_t)block_sum_f((float)n_finite, sh);      // counts up to 2^18 per row: exact in fp32
    if (finite == 0) {
        if (tid == 0) {
            *out_token = 0xFFFFFFFFu;
            *out_prob = 0.0f;
        }
        return;
    }
    const uint32_t want = min(k, finite);                      // fewer finite entries than top_k: all of them
    find_bin(sh, 2048, want);
    const uint32_t b1 = sh.bin, above1 = sh.above;
    __syncthreads();
    for (uint32_t b = tid; b < 2048; b += kSampleThreads) sh.hist[b] = 0;
    __syncthreads();
    for (uint32_t i = tid; i < count; i += kSampleThreads) {
        const float c = sample_capped(row[i], cap);
        if (c == -INFINITY) continue;
        const uint32_t q = sample_key(c);
        if ((q >> 21) == b1) atomicAdd(&sh.hist[(q >> 10) & 2047u], 1u);
    }
    find_bin(sh, 2048, want - above1);
    const uint32_t b2 = sh.bin, above2 = above1 + sh.above;
    __syncthreads();
    for (uint32_t b = tid; b < 1024; b += kSampleThreads) sh.hist[b] = 0;
    __syncthreads();
    const uint32_t top22 = (b1 << 11) | b2;
    for (uint32_t i = tid; i < count; i += kSampleThreads) {
        const float c = sample_capped(row[i], cap);
        if (c == -INFINITY) continue;
        const uint32_t q = sample_key(c);
        if ((q >> 10) == top22) atomicAdd(&sh.hist[q & 1023u], 1u);
    }
    find_bin(sh, 1024, want - above2);
    const uint32_t threshold = (top22 << 10) | sh.bin;         // the key of the want-th largest capped logit
    const uint32_t above = above2 + sh.above, need = want - above;     // `need` of the entries equal to it, lowest indices first
    __syncthreads();

    // ---- gather: everything above the threshold, and per wave the first `need` indices equal to it -----------
    // wave w walks the contiguous piece [w * piece, (w + 1) * piece) of the row 64 entries at a time, so a ballot's
    // bit order is index order
    const uint32_t piece = ((count + kSampleWaves - 1) / kSampleWaves + 63) / 64 * 64;
    uint32_t eq_seen = 0;
    for (uint32_t base = wave * piece; base < min(count, (wave + 1) * piece); base += 64) {
        const uint32_t i = base + lane;
        float c = -INFINITY;
        if (i < count) c = sample_capped(row[i], cap);
        const uint32_t q = c == -INFINITY ? 0u : sample_key(c);
        if (q > threshold) {
            const uint32_t slot = atomicAdd(&sh.n_above, 1u);
            sh.cand_v[slot] = c;                                // fewer than want <= 256 of them
            sh.cand_i[slot] = i;
        }
        const bool eq = c != -INFINITY && q == threshold;
        const unsigned long long mask = __ballot(eq);
        if (eq) {
            const uint32_t rank = eq_seen + __popcll(mask & ((1ull << lane) - 1ull));
            if (rank < need) sh.wave_eq[wave][rank] = i;
        }
        eq_seen += __popcll(mask);
    }
    if (lane == 0) sh.wave_eq_n[wave] = min(eq_seen, need);
    __syncthreads();
    // the equal entries in index order: wave 0's first, then wave 1's, ... until `need` are placed
    if (tid < need) {
        uint32_t skip = tid, w = 0;
        while (w < (uint32_t)kSampleWaves && skip >= sh.wave_eq_n[w]) skip -= sh.wave_eq_n[w++];
        const uint32_t i = sh.wave_eq[w][skip];                // exists: the waves hold at least `need` together
        sh.cand_v[above + tid] = sample_capped(row[i], cap);
        sh.cand_i[above + tid] = i;
    }
    __syncthreads();
    const uint32_t n = want;
    // ---- rank the candidates: larger value first, then lower index (sample_before, logit.metal:1059-1062) -----
    if (tid < n) {
        const float v = sh.cand_v[tid];
        const uint32_t i = sh.cand_i[tid];
        uint32_t rank = 0;
        for (uint32_t u = 0; u < n; ++u) {
            const float vu = sh.cand_v[u];
            const uint32_t iu = sh.cand_i[u];
            rank += (vu > v || (vu == v && iu < i)) ? 1u : 0u;
        }
        sh.sorted_v[rank] = v;
        sh.sorted_i[rank] = i;
    }
    __syncthreads();
    sample_finish(sh, p, n, total1, seed, key, ids, out_token, out_prob);
}

__device__ __forceinline__ uint32_t sample_position_key(const SampleRule &p, const uint32_t *__restrict__ key_offset, uint32_t r) {
    return p.key_base + (key_offset ? key_offset[0] : 0u) + r;
}

__global__ __launch_bounds__(kSampleThreads) void sample_rows_kernel(const float *__restrict__ logits, uint32_t stride, uint32_t count,
                                                                     const uint32_t *__restrict__ ids, SampleRule p,
                                                                     const uint32_t *__restrict__ key_offset,
                                                                     uint32_t *__restrict__ out_tokens, float *__restrict__ out_prob) {
    __shared__ SampleShared sh;
    const uint32_t r = blockIdx.x;
    sample_one_row(sh, logits + (size_t)r * stride, count, ids, p, sample_position_key(p, key_offset, r), out_tokens + r, out_prob + r);
}

// ---- long rows: one sweep by many blocks, then one block per row -------------------------------------------------
// Bound: the sweep is instruction issue (one tanhf and one expf, or the noise's two logf and 64-bit products, per logit),
// spread over 128 blocks per full-vocabulary row; the second launch is a chain of round trips to memory and LDS, which is why its
// reductions are register moves: 262,144 logits, the 64 largest, 5.2 + 12.1 us with shuffles and the bound found bit by bit, then 4.6 +
// 9.8, now 4.6 + 8.2: a wave takes its places in a list with one atomic (one per slot: 1.1 us), the raw bound is one wave's, the running sum
// of the shares register moves with the noise beside it. The stages then, of 8.2: keys and sums 1.2, bound 2.0, list 0.8, candidates 1.6, caps
// and ranks 0.9, draw 0.9.
static_assert(kSampleMaxSegments <= kSampleThreads, "the finishing launches bring one segment per thread");
constexpr int kScanThreads = 256, kScanPer = kSampleSegment / kScanThreads;
static_assert(kSampleSegment % kScanThreads == 0 && kSampleGroup == 64, "a wave's load is one group");

// TRUNCATED: every 64-wide group's largest capped logit as its key (0: nothing finite) and the block's share of the
// T = 1 normaliser. Else: the block's largest capped logit, its tempered sum relative to that and its winner of the draw.
template <bool TRUNCATED>
__global__ __launch_bounds__(kScanThreads) void sample_scan_kernel(const float *__restrict__ logits, uint32_t stride, uint32_t count,
                                                                   const uint32_t *__restrict__ ids, SampleRule p,
                                                                   const uint32_t *__restrict__ key_offset, SampleScratch sc) {
    __shared__ float s_f[kScanThreads / 64];
    __shared__ uint32_t s_n[kScanThreads / 64];
    __shared__ unsigned long long s_k[kScanThreads / 64];
    const uint32_t r = blockIdx.y, seg = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const float *row = logits + (size_t)r * stride;
    const float cap = p.softcap;
    float c[kScanPer];
#pragma unroll
    for (int u = 0; u < kScanPer; ++u) {
        const uint32_t i = seg * kSampleSegment + u * kScanThreads + tid;
        c[u] = i < count ? row[i] : -INFINITY;
    }
#pragma unroll
    for (int u = 0; u < kScanPer; ++u) c[u] = sample_capped(c[u], cap);
    if constexpr (TRUNCATED) {
        float sum = 0.0f;
        uint32_t finite = 0;
        uint32_t top[kScanPer];
#pragma unroll
        for (int u = 0; u < kScanPer; ++u) {
            top[u] = c[u] == -INFINITY ? 0u : sample_key(c[u]);
            if (c[u] != -INFINITY) {
                sum += expf(c[u] - cap);
                ++finite;
            }
        }
#pragma unroll
        for (int u = 0; u < kScanPer; ++u) top[u] = wave_max_u32(top[u]);
        sum = wave_butterfly_sum(sum);
        finite = (uint32_t)wave_butterfly_sum((float)finite);
        uint32_t *keys = sc.group_keys + (size_t)r * kSampleMaxGroups + seg * (kSampleSegment / kSampleGroup);
#pragma unroll
        for (int u = 0; u < kScanPer; ++u)
            if (lane == 0) keys[u * (kScanThreads / 64) + wave] = top[u];
        if (lane == 0) {
            s_f[wave] = sum;
            s_n[wave] = finite;
        }
        __syncthreads();
        if (tid == 0) {
            SampleSegment out{};
            for (int w = 0; w < kScanThreads / 64; ++w) {
                out.sum += s_f[w];
                out.finite += s_n[w];
            }
            sc.segments[(size_t)r * kSampleMaxSegments + seg] = out;
        }
    } else {
        const float invT = 1.0f / p.temperature;
        const uint32_t key = sample_position_key(p, key_offset, r);
        const unsigned long long seed = ((unsigned long long)p.seed_hi << 32) | p.seed_lo;
        float m = -INFINITY;
#pragma unroll
        for (int u = 0; u < kScanPer; ++u) m = fmaxf(m, c[u]);
        m = wave_max_f32(m);
        if (lane == 0) s_f[wave] = m;
        __syncthreads();
        for (int w = 0; w < kScanThreads / 64; ++w) m = fmaxf(m, s_f[w]);
        __syncthreads();
        float sum = 0.0f;
        unsigned long long best = 0ull;
#pragma unroll
        for (int u = 0; u < kScanPer; ++u) {
            if (c[u] == -INFINITY) continue;
            const uint32_t i = seg * kSampleSegment + u * kScanThreads + tid;
            sum += expf((c[u] - m) * invT);
            const float g = c[u] * invT + sample_gumbel(seed, key, ids ? ids[i] : i);
            const unsigned long long k = ((unsigned long long)sample_key(g) << 32) | (0xFFFFFFFFu - i);
            best = k > best ? k : best;
        }
        sum = wave_butterfly_sum(sum);
        best = wave_max_key(best);
        if (lane == 0) {
            s_f[wave] = sum;
            s_k[wave] = best;
        }
        __syncthreads();
        if (tid == 0) {
            SampleSegment out{};
            out.top = m;
            for (int w = 0; w < kScanThreads / 64; ++w) {
                out.sum += s_f[w];
                out.best = s_k[w] > out.best ? s_k[w] : out.best;
            }
            sc.segments[(size_t)r * kSampleMaxSegments + seg] = out;
        }
    }
}

// Without truncation: the segments' winners and sums merged, one block per row.
__global__ __launch_bounds__(kSampleThreads) void sample_merge_kernel(const float *__restrict__ logits, uint32_t stride, uint32_t n_seg,
                                                                          SampleRule p, SampleScratch sc, uint32_t *__restrict__ out_tokens,
                                                                          float *__restrict__ out_prob) {
    __shared__ SampleShared sh;
    const uint32_t r = blockIdx.x, tid = threadIdx.x;
    const float invT = 1.0f / p.temperature;
    SampleSegment mine{};
    mine.top = -INFINITY;
    if (tid < n_seg) mine = sc.segments[(size_t)r * kSampleMaxSegments + tid];
    const float m = block_max_f(mine.top, sh);
    const float total = block_sum_f(mine.best ? mine.sum * expf((mine.top - m) * invT) : 0.0f, sh);
    const unsigned long long best = block_max_k(mine.best, sh);
    if (tid == 0) {
        const uint32_t j = best ? 0xFFFFFFFFu - (uint32_t)best : 0xFFFFFFFFu;
        out_tokens[r] = j;
        out_prob[r] = (j == 0xFFFFFFFFu || !(total > 0.0f)) ? 0.0f
                                                            : expf((sample_capped(logits[(size_t)r * stride + j], p.softcap) - m) * invT) / total;
    }
}

// With truncation: the bound from the groups' maxima, the candidates of the groups that reach it, the exact ranking.
constexpr int kPickSlots = kSampleMaxGroups / kSampleThreads;
constexpr uint32_t kPickMaxGroups = 1024, kPickMaxCands = 1024;

__global__ __launch_bounds__(kSampleThreads) void sample_pick_kernel(const float *__restrict__ logits, uint32_t stride, uint32_t count,
                                                                     uint32_t n_seg, const uint32_t *__restrict__ ids, SampleRule p,
                                                                     const uint32_t *__restrict__ key_offset, SampleScratch sc,
                                                                     uint32_t *__restrict__ out_tokens, float *__restrict__ out_prob) {
    __shared__ SampleShared sh;
    __shared__ __align__(16) unsigned long long cand[kPickMaxCands];          // key << 32 | ~index: larger value first, then lower index
    __shared__ uint32_t group_list[kPickMaxGroups];
    __shared__ uint32_t n_list, n_cand, reach_of[2][kSampleWaves];
    const uint32_t r = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const float *row = logits + (size_t)r * stride;
    const uint32_t n_groups = n_seg * (kSampleSegment / kSampleGroup);       // groups past the row's end hold key 0
    uint32_t keys[kPickSlots];
#pragma unroll
    for (int s = 0; s < kPickSlots; ++s) {
        const uint32_t g = s * kSampleThreads + tid;
        keys[s] = g < n_groups ? sc.group_keys[(size_t)r * kSampleMaxGroups + g] : 0u;
    }
    SampleSegment mine{};
    if (tid < n_seg) mine = sc.segments[(size_t)r * kSampleMaxSegments + tid];
    if (tid == 0) n_list = n_cand = 0;
    cand[tid] = 0ull;
    const float2 sums = block_sum_f2(make_float2(mine.sum, (float)mine.finite), sh);
    const float total1 = sums.x;
    const uint32_t finite = (uint32_t)sums.y;                    // at most 2^19: exact in fp32
    if (finite == 0) {
        if (tid == 0) {
            out_tokens[r] = 0xFFFFFFFFu;
            out_prob[r] = 0.0f;
        }
        return;
    }
    const uint32_t want = min(p.top_k, finite);
    // A bound that at least `want` groups reach, found on the threads' largest keys (a lower bound of the groups' own want-th
    // largest), four bits at a time from the top until it leaves out most of the others: each of the sixteen waves counts for one
    // value of the four, from the first bits in which any two differ. (Bit by bit by one wave it was 2 of the launch's 11.5 us.)
    uint32_t most = 0;
#pragma unroll
    for (int s = 0; s < kPickSlots; ++s) most = max(most, keys[s]);
    sh.hist[tid] = most;
    __syncthreads();
    static_assert(kSampleWaves == 16, "a wave per value of four bits");
    uint32_t held[kSampleWaves];
#pragma unroll
    for (int s = 0; s < kSampleWaves; ++s) held[s] = sh.hist[64 * s + lane];
    // the bits that all of them share need no counting (a row's largest values have their upper eight or so in common)
    const uint32_t one = (uint32_t)__builtin_amdgcn_readfirstlane((int)held[0]);
    uint32_t differ = 0, reach = kSampleThreads;
#pragma unroll
    for (int s = 0; s < kSampleWaves; ++s) differ |= held[s] ^ one;
    differ = wave_max_u32(differ);                              // its highest bit is the highest in which any two differ
    const int top = differ ? (31 - __builtin_clz(differ)) & ~3 : -4;
    uint32_t low = top < 28 ? one >> (top + 4) << (top + 4) : 0u;
#pragma unroll 1
    for (int shift = top; shift >= 0 && reach > want + want / 2; shift -= 4) {
        const uint32_t at = low | (wave << shift);
        uint32_t c = 0;
#pragma unroll
        for (int s = 0; s < kSampleWaves; ++s) c += __popcll(__ballot(held[s] >= at));
        uint32_t *const counts = reach_of[(shift >> 2) & 1];
        if (lane == 0) counts[wave] = c;
        __syncthreads();
        c = counts[lane & 15];                                  // (wave 0's value is the bound so far: at least `want` reach it)
        const int most_of = 31 - __builtin_clz((uint32_t)__ballot(c >= want) & 0xFFFFu);
        low |= (uint32_t)most_of << shift;
        reach = (uint32_t)__builtin_amdgcn_readlane((int)c, most_of);
    }
    const uint32_t bound = max(low, 1u);           // fewer finite groups than `want`: every finite logit is a candidate
    const uint32_t key = sample_position_key(p, key_offset, r);
    // The candidates are first told apart by their raw value: `raw_low` is below every logit whose capped value reaches the
    // bound (the inverse of the cap at the bound less a few thousand times tanhf's error), so that the cap itself is
    // computed once per candidate and not for the other 63 logits of its group.
    // (One wave makes it for all, beside the others' lists.)
    if (wave == kSampleWaves - 1) {
        float low_of = -FLT_MAX;
        if (bound > 1u) {
            const float at = __uint_as_float((bound & 0x80000000u) ? (bound & 0x7FFFFFFFu) : ~bound) / p.softcap;
            const float z = fminf(at - 1e-4f * fabsf(at) - 1e-6f, 0.9999f);
            if (z > -0.9999f) low_of = p.softcap * atanhf(z);
        }
        if (lane == 0) sh.red_f[0] = low_of;
    }
    // (a wave takes its places in a list all at once: one after the other the counter's answers were a chain of round trips to LDS)
    {
        unsigned long long mask[kPickSlots];
        uint32_t n = 0;
#pragma unroll
        for (int s = 0; s < kPickSlots; ++s) mask[s] = __ballot(keys[s] >= bound), n += (uint32_t)__popcll(mask[s]);
        if (n) {
            uint32_t first = 0;
            if (lane == 0) first = atomicAdd(&n_list, n);
            first = (uint32_t)__builtin_amdgcn_readfirstlane((int)first);
#pragma unroll
            for (int s = 0; s < kPickSlots; ++s) {
                if (mask[s] == 0ull) continue;
                const uint32_t place = first + lanes_in_front(mask[s]);
                if (keys[s] >= bound && place < kPickMaxGroups) group_list[place] = s * kSampleThreads + tid;
                first += (uint32_t)__popcll(mask[s]);
            }
        }
    }
    __syncthreads();
    const uint32_t listed = n_list;
    const float raw_low = sh.red_f[0];
    bool fits = listed <= kPickMaxGroups;
    if (fits) {
        constexpr int kAhead = 8;
        for (uint32_t base = wave; base < listed; base += kAhead * kSampleWaves) {
            float v[kAhead];
            uint32_t at[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const uint32_t li = base + u * kSampleWaves;
                at[u] = li < listed ? group_list[li] * kSampleGroup + lane : 0xFFFFFFFFu;
                v[u] = at[u] < count ? row[at[u]] : NAN;
            }
            unsigned long long mask[kAhead];
            uint32_t n = 0;
#pragma unroll
            for (int u = 0; u < kAhead; ++u) mask[u] = __ballot(v[u] >= raw_low && v[u] <= FLT_MAX), n += (uint32_t)__popcll(mask[u]);
            if (n == 0) continue;
            uint32_t first = 0;
            if (lane == 0) first = atomicAdd(&n_cand, n);
            first = (uint32_t)__builtin_amdgcn_readfirstlane((int)first);
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                if (mask[u] == 0ull) continue;
                const uint32_t place = first + lanes_in_front(mask[u]);
                if ((mask[u] >> lane & 1ull) && place < kPickMaxCands) cand[place] = ((unsigned long long)__float_as_uint(v[u]) << 32) | (0xFFFFFFFFu - at[u]);
                first += (uint32_t)__popcll(mask[u]);
            }
        }
        __syncthreads();
        fits = fits && n_cand <= kPickMaxCands;
    }
    if (!fits) {      // more ties at the bound than the lists hold
        __syncthreads();
        sample_one_row(sh, row, count, ids, p, key, out_tokens + r, out_prob + r);
        return;
    }
    const uint32_t n = n_cand;
    static_assert(kPickMaxCands == (uint32_t)kSampleThreads && kPickMaxCands % 4 == 0, "one candidate per thread");
    if (tid < n) {
        const unsigned long long raw = cand[tid];
        const uint32_t q = sample_key(sample_capped(__uint_as_float((uint32_t)(raw >> 32)), p.softcap));
        cand[tid] = q >= bound ? ((unsigned long long)q << 32) | (uint32_t)raw : 0ull;
    }
    // rank by counting: the threads of a candidate share the comparisons, four keys per read (all keys differ: they carry
    // the index; the list ends in zeros)
    const uint32_t parts = max(1u, (uint32_t)kSampleThreads / n), per = ((n + parts - 1) / parts + 3) & ~3u;
    uint32_t *rank_of = sh.hist;
    if (tid < n) rank_of[tid] = 0;
    __syncthreads();
    const uint32_t ci = tid % n, part = tid / n;
    if (part < parts) {
        const unsigned long long own = cand[ci];
        uint32_t rank = 0;
        for (uint32_t u = part * per; u < min(n, (part + 1) * per); u += 4) {
            const ulonglong2 a = *reinterpret_cast<const ulonglong2 *>(&cand[u]), b = *reinterpret_cast<const ulonglong2 *>(&cand[u + 2]);
            rank += (a.x > own ? 1u : 0u) + (a.y > own ? 1u : 0u) + (b.x > own ? 1u : 0u) + (b.y > own ? 1u : 0u);
        }
        if (rank) atomicAdd(&rank_of[ci], rank);
    }
    __syncthreads();
    if (tid < n && rank_of[tid] < want && cand[tid]) {
        const unsigned long long own = cand[tid];
        const uint32_t q = (uint32_t)(own >> 32), rank = rank_of[tid];
        sh.sorted_v[rank] = __uint_as_float((q & 0x80000000u) ? (q & 0x7FFFFFFFu) : ~q);
        sh.sorted_i[rank] = 0xFFFFFFFFu - (uint32_t)own;
    }
    sample_finish(sh, p, want, total1, ((unsigned long long)p.seed_hi << 32) | p.seed_lo, key, ids, out_tokens + r, out_prob + r);
}

}  // namespace

// The sweep by many blocks: rows long enough to fill several blocks, with at least twice as many groups as survivors (so that
// the bound leaves out most of the row), and no longer than the scratch holds groups for.
bool sample_takes_scratch(uint32_t count, uint32_t top_k) {
    const bool truncated = top_k > 0u && top_k < count;
    return count >= max(4096u, truncated ? 2u * kSampleGroup * top_k : 0u) && count <= kSampleMaxGroups * kSampleGroup;
}

hipError_t launch_sample_rows(hipStream_t s, const float *logits, uint32_t stride, uint32_t rows, uint32_t count,
                              const uint32_t *ids, float temperature, float top_p, uint32_t top_k, uint32_t key_base,
                              float softcap, unsigned long long seed, const uint32_t *key_offset, uint32_t *out_tokens,
                              float *out_prob, SampleScratch sc) {
    const SampleRule rule{temperature, top_p, top_k, key_base, softcap, (uint32_t)seed, (uint32_t)(seed >> 32)};
    const bool truncated = top_k > 0u && top_k < count;
    const bool use_scan = sc.group_keys && sample_takes_scratch(count, top_k);
    if (use_scan) {
        const uint32_t n_seg = (count + kSampleSegment - 1) / kSampleSegment;
        const dim3 grid(n_seg, rows);
        if (truncated) {
            hipLaunchKernelGGL(sample_scan_kernel<true>, grid, dim3(kScanThreads), 0, s, logits, stride, count, ids, rule, key_offset, sc);
            hipLaunchKernelGGL(sample_pick_kernel, dim3(rows), dim3(kSampleThreads), 0, s, logits, stride, count, n_seg, ids, rule, key_offset,
                               sc, out_tokens, out_prob);
        } else {
            hipLaunchKernelGGL(sample_scan_kernel<false>, grid, dim3(kScanThreads), 0, s, logits, stride, count, ids, rule, key_offset, sc);
            hipLaunchKernelGGL(sample_merge_kernel, dim3(rows), dim3(kSampleThreads), 0, s, logits, stride, n_seg, rule, sc, out_tokens, out_prob);
        }
        return hipGetLastError();
    }
    hipLaunchKernelGGL(sample_rows_kernel, dim3(rows), dim3(kSampleThreads), 0, s, logits, stride, count, ids, rule, key_offset,
                       out_tokens, out_prob);
    return hipGetLastError();
}

}  // namespace ffmoe
