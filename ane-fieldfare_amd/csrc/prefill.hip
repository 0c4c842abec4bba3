// Prefill routed experts: expert-sorted (token, expert) pairs, then two grouped GEMMs on the matrix
// units whose weight tiles are dequantised INT4 -> bf16 on the way into their operands.
//
// Replaces the host-side pair sort of PrefillMoEGrouping.groupTokenExpertPairs
// (Kernels/Prefill/MoE/PrefillMoEGrouping.swift:49-110), prefill_routed_gate_up_tensorops /
// prefill_routed_down_tensorops (Metal/Prefill/prefill.metal:609-779) and the ANE guest
// (Runtime/Inference/ANERoutedPrefillBackend.swift:348-427, Metal/ANE/ane_prefill.metal).
//
// Sort: a stable counting sort keyed by expert. Items keep their input order inside an expert, so
// routes taken from the router's [token][rank] table come out in (expert, token, rank) order - the
// order the reference's comparator produces (PrefillMoEGrouping.swift:66-75). Only integer counting uses
// LDS atomics; every position comes from prefix sums, so the result does not depend on timing.
//
// GEMM: items of one M-tile of up to 256 same-expert pairs x 256 weight rows, one or two blocks per compute unit walking lists of them. Every
// wave expands its own arena tile to bf16(fma(q, scale, bias)) - the reference's 16-bit tile weight (prefill.metal:581-590) - in
// the register layout v_mfma_f32_16x16x32_bf16 wants; the pairs' inputs and the packed tiles go from global memory straight into LDS.
// fp32 accumulation; GELU-tanh(gate) * up in the epilogue.
// bf16 activations make the reference's power-of-two block scaling (prefill.metal:593-598, an FP16 range
// fix) unnecessary.
#include "common.hpp"
#include "kernels.hpp"
#include "stream.hpp"

namespace ffmoe {
namespace {

constexpr int kSortBlock = 256;
// Pairs per M-tile, a multiple of 16 up to kBM, and what divides by it: n * `divide` >> 32 is n / rows for every n where rows is a
// power of two, and up to 2^24 otherwise.
struct TileRows {
    uint32_t rows, divide;
    __host__ __device__ explicit TileRows(uint32_t r) : rows(r), divide((uint32_t)(((1ull << 32) + r - 1) / r)) {}
    __device__ __forceinline__ uint32_t whole(uint32_t n) const { return __umulhi(n, divide); }
};
constexpr int kBM = FFMOE_PREFILL_TILE_M;   // pairs per M-tile
constexpr int kTilesPerBlock = 4;           // arena tiles (of 16 + 16 rows) per N-block

// ---------------------------------------------------------------------------------------------------
// Item sources: a router table [t][top_k] (item = route) or an explicit pair list.
// ---------------------------------------------------------------------------------------------------
struct ItemSource {
    const uint32_t *idx;       // router table: expert per route, or nullptr
    const uint16_t *w;         // router table: weight bits per route
    const ffmoe_pair *pairs;   // explicit pairs, or nullptr
    uint32_t n_items;
    uint32_t top_k;
    uint32_t n_experts;
    uint32_t t;
};

__device__ __forceinline__ uint32_t item_expert(const ItemSource &src, uint32_t i) {
    if (i >= src.n_items) return 0xFFFFFFFFu;
    if (src.pairs) {
        const ffmoe_pair p = src.pairs[i];
        return (p.expert < src.n_experts && p.token < src.t && p.rank < src.top_k) ? p.expert : 0xFFFFFFFFu;
    }
    const uint32_t e = src.idx[i];
    // zero-weight routes are dropped, as the reference's prefill does (RealForwardRunner.swift:1528-1530)
    return ((src.w[i] & 0x7FFFu) != 0 && e < src.n_experts) ? e : 0xFFFFFFFFu;
}

__global__ __launch_bounds__(kSortBlock) void prefill_hist_kernel(ItemSource src, uint32_t *__restrict__ block_cnt) {
    __shared__ uint32_t cnt[FFMOE_MAX_EXPERTS];
    cnt[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t e = item_expert(src, blockIdx.x * kSortBlock + threadIdx.x);
    if (e != 0xFFFFFFFFu) atomicAdd(&cnt[e], 1u);
    __syncthreads();
    if (threadIdx.x < src.n_experts) block_cnt[(size_t)blockIdx.x * src.n_experts + threadIdx.x] = cnt[threadIdx.x];
}

// One block of 1024 threads: per expert, turn the per-block counts into per-block bases, then lay out the
// experts one after the other and cut each into M-tiles. Thread (expert e, chunk c) owns a contiguous run
// of sort blocks, so the counts of a whole column are in flight at once and - up to kScanKeep per thread -
// stay in registers between the summing pass and the pass that writes the bases.
constexpr int kScanThreads = 1024;
// (kScanKeep: 16, or 32 where a thread's run is longer - 8,192 rows x 8 routes with 128 experts: 15.4 -> 10.3 us, the second half of
// a run was read twice; short runs pay for the longer unrolled passes, 443.1 against 441.4 us for a plugin chunk of 3,079 rows)

template <int kScanKeep>
__global__ __launch_bounds__(kScanThreads) void prefill_scan_kernel(uint32_t n_blocks, uint32_t n_experts, uint32_t e_pad,
                                                                    uint32_t *__restrict__ block_cnt,
                                                                    PrefillPlan *__restrict__ plan,
                                                                    PrefillTile *__restrict__ tiles, uint32_t max_tiles,
                                                                    TileRows bm) {
    __shared__ uint32_t total[FFMOE_MAX_EXPERTS], last_rows[FFMOE_MAX_EXPERTS];    // pairs, and those past the whole tiles
    __shared__ uint32_t offset[FFMOE_MAX_EXPERTS + 1];
    __shared__ uint32_t tile_off[FFMOE_MAX_EXPERTS + 1];
    __shared__ uint32_t part[kScanThreads];                 // [chunk][e_pad]: chunk sums, then chunk bases
    __shared__ unsigned long long scan_own[FFMOE_MAX_EXPERTS], wave_sum[FFMOE_MAX_EXPERTS / 64];
    __shared__ uint32_t wave_live[FFMOE_MAX_EXPERTS / 64];
    __shared__ uint32_t shorter[3][FFMOE_MAX_EXPERTS];      // per expert: shorter tiles in all, in front of it, ranked above its own
    const uint32_t e = threadIdx.x % e_pad, ch = threadIdx.x / e_pad, chunks = kScanThreads / e_pad;
    const uint32_t per = (n_blocks + chunks - 1) / chunks;
    const uint32_t b_lo = min(n_blocks, ch * per), b_hi = min(n_blocks, b_lo + per);
    const bool live = e < n_experts;
    uint32_t keep[kScanKeep];
    uint32_t sum = 0;
#pragma unroll
    for (int u = 0; u < kScanKeep; ++u) {
        keep[u] = live && b_lo + u < b_hi ? block_cnt[(size_t)(b_lo + u) * n_experts + e] : 0;
        sum += keep[u];
    }
    if (live)
        for (uint32_t b = b_lo + kScanKeep; b < b_hi; ++b) sum += block_cnt[(size_t)b * n_experts + e];
    part[threadIdx.x] = sum;
    if (threadIdx.x < FFMOE_MAX_EXPERTS) {
        total[threadIdx.x] = 0;
        shorter[0][threadIdx.x] = shorter[1][threadIdx.x] = shorter[2][threadIdx.x] = 0;
    }
    __syncthreads();
    if (ch == 0 && live) {
        uint32_t run = 0;
        for (uint32_t c = 0; c < min(chunks, n_blocks); ++c) {      // (the chunks behind hold nothing)
            const uint32_t v = part[c * e_pad + e];
            part[c * e_pad + e] = run;
            run += v;
        }
        total[e] = run;
    }
    __syncthreads();
    // exclusive prefix sums over the experts of (pairs, tiles), packed into one 64-bit value: four waves scan 64
    // experts each, then add the waves in front of them
    if (threadIdx.x < FFMOE_MAX_EXPERTS) {
        const uint32_t i = threadIdx.x, lane = i & 63, wv = i >> 6;
        const uint32_t n = i < n_experts ? total[i] : 0;
        const uint32_t whole = bm.whole(n), rest = n - whole * bm.rows;
        last_rows[i] = rest;
        const unsigned long long own = ((unsigned long long)(whole + (rest != 0 ? 1u : 0u)) << 32) | n;
        unsigned long long inc = own;
#pragma unroll
        for (int sh = 1; sh < 64; sh <<= 1) {
            const unsigned long long up = __shfl_up(inc, sh, 64);
            if (lane >= (uint32_t)sh) inc += up;
        }
        const uint32_t with_pairs = (uint32_t)__popcll(__ballot(n != 0));
        if (lane == 63) wave_sum[wv] = inc, wave_live[wv] = with_pairs;
        scan_own[i] = inc - own;
    }
    __syncthreads();
    if (threadIdx.x < FFMOE_MAX_EXPERTS) {
        const uint32_t i = threadIdx.x, wv = i >> 6;
        unsigned long long base = 0;
        for (uint32_t v = 0; v < wv; ++v) base += wave_sum[v];
        const unsigned long long ex = base + scan_own[i];
        if (i <= n_experts) {
            offset[i] = (uint32_t)ex;
            tile_off[i] = (uint32_t)(ex >> 32);
        }
        if (i == n_experts || (i == FFMOE_MAX_EXPERTS - 1 && n_experts == FFMOE_MAX_EXPERTS)) {
            // the totals: the prefix in front of the first expert past the end (or, with every slot in use, the last
            // expert's prefix plus its own share)
            unsigned long long all = ex;
            if (i != n_experts) {
                const uint32_t n = total[i];
                all += ((unsigned long long)(bm.whole(n) + (last_rows[i] != 0 ? 1u : 0u)) << 32) | n;
                offset[n_experts] = (uint32_t)all;
                tile_off[n_experts] = (uint32_t)(all >> 32);
            }
            plan->n_pairs = (uint32_t)all;
            plan->n_tiles = min((uint32_t)(all >> 32), max_tiles);
            plan->live_experts = wave_live[0] + wave_live[1] + wave_live[2] + wave_live[3];
            plan->expert_offset[n_experts] = (uint32_t)all;
        }
    }
    __syncthreads();
    // The tile list runs from the largest tile down: the full tiles in expert order, then every expert's last, shorter
    // tile by its rows (ties in expert order). The GEMM grids walk the list eight tiles at a time, so the launches end
    // with their shortest blocks instead of with whatever the last experts hold (a Zipf chunk's heavy experts sit
    // anywhere in the expert order). Where an expert's shorter tile goes takes a look at every other expert's: the
    // threads of an expert share that out (one thread alone is a chain of two thousand instructions).
    if (live) {
        const uint32_t rest = last_rows[e], per_o = (e_pad + chunks - 1) / chunks;
        const uint32_t o_lo = min(e_pad, ch * per_o), o_hi = min(e_pad, o_lo + per_o);
        uint32_t all = 0, in_front = 0, above = 0;
        for (uint32_t o = o_lo; o < o_hi; ++o) {
            const uint32_t r = last_rows[o];                   // experts past n_experts hold zero
            const uint32_t has = r != 0 ? 1u : 0u;
            all += has;
            in_front += has & (o < e ? 1u : 0u);
            above += has & ((r > rest || (r == rest && o < e)) ? 1u : 0u);
        }
        if (all) {
            atomicAdd(&shorter[0][e], all);
            atomicAdd(&shorter[1][e], in_front);
            atomicAdd(&shorter[2][e], above);
        }
    }
    __syncthreads();
    if (!live) return;
    uint32_t run = offset[e] + part[threadIdx.x];
#pragma unroll
    for (int u = 0; u < kScanKeep; ++u) {
        if (b_lo + u < b_hi) block_cnt[(size_t)(b_lo + u) * n_experts + e] = run;      // count -> base, in place
        run += keep[u];
    }
    for (uint32_t b = b_lo + kScanKeep; b < b_hi; ++b) {
        const uint32_t c = block_cnt[(size_t)b * n_experts + e];
        block_cnt[(size_t)b * n_experts + e] = run;
        run += c;
    }
    if (ch != 0) return;
    plan->expert_offset[e] = offset[e];
    plan->expert_count[e] = total[e];
    // a tile keeps its number in row order, which places its activation blocks
    const uint32_t n_full = bm.whole(total[e]), nt = n_full + (last_rows[e] != 0 ? 1u : 0u);
    const uint32_t shorter_tiles = shorter[0][e], shorter_in_front = shorter[1][e], ranked_above = shorter[2][e];
    const uint32_t full_in_front = tile_off[e] - shorter_in_front, full_tiles = tile_off[n_experts] - shorter_tiles;
    for (uint32_t i = 0; i < nt; ++i) {
        const uint32_t ti = i < n_full ? full_in_front + i : full_tiles + ranked_above;
        if (ti < max_tiles) {
            PrefillTile tl;
            tl.expert = e;
            tl.row_start = offset[e] + i * bm.rows;
            tl.rows = min(bm.rows, total[e] - i * bm.rows);
            tl.order = tile_off[e] + i;
            tiles[ti] = tl;
        }
    }
}

// The lanes of the wave whose item has this lane's expert: a mask built from one ballot per bit of the expert number.
__device__ __forceinline__ unsigned long long same_expert(uint32_t e) {
    static_assert(FFMOE_MAX_EXPERTS <= 256, "eight ballots tell the experts apart");
    unsigned long long same = __ballot(e != 0xFFFFFFFFu);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const bool bit = (e >> b) & 1u;
        const unsigned long long with = __ballot(bit);
        same &= bit ? with : ~with;
    }
    return same;
}

__device__ __forceinline__ void place_item(const ItemSource &src, uint32_t i, uint32_t pos, uint32_t *__restrict__ sorted_token,
                                           uint32_t *__restrict__ sorted_out_row) {
    uint32_t token, out_row;
    if (src.pairs) {
        const ffmoe_pair p = src.pairs[i];
        token = p.token;
        out_row = p.token * src.top_k + p.rank;
    } else {
        token = i / src.top_k;
        out_row = i;
    }
    sorted_token[pos] = token;
    sorted_out_row[pos] = out_row;
}

// The three kernels' work in one launch, a block per expert: every block counts all items in LDS, marks its own expert's as it goes,
// and knows after that where its expert's pairs and tiles begin - sums over the counts, no block waits for another. Wave w of a
// block has a contiguous run of items, 64 at a time, eight loads in flight; an item's place is its expert's beginning and what its wave
// and the waves in front hold of it. Same order as the three.
// Bound: few items, latencies one behind the other; many, the counting, 27 cycles for a wave's 64 items, which every block does anew.
// Call of a layer of 64 x 64, top-8 of 128, us: up to 3,072 items one block did the three kernels' work, that | this: 296 items 16.8 |
// 14.3, 2,408 items 20.2 | 16.8; beyond, the three | this: 4,096 items 22.5 | 17.6, 8,000 items 23.6 | 17.7, 16,000 items 25.2 | 21.1,
// 24,576 items 27.5 | 25.0 (Zipf routes 28.9 | 26.6), 32,768 items 28.9 | 29.3, 65,536 items 40 | 48; top-8 of 256, whose scan is
// longer, 24,576 items 33.3 | 25.7, 65,536 items 57 | 47; top-1 of 32, 16,000 items 23.5 | 20.9, 24,576 items 25.4 | 25.9. Without the
// shared start (blocks that begin at items of their own): the same.
constexpr int kSortRuns = 64;                               // items of a lane: a bit each
// Up to how many items one launch sorts: where it crosses the three, later with skewed tables (whose lanes meet at the three launches'
// counters too) than with uniform ones, earlier with lists in order (which cost the three few turns). Three | one, us: lists, top-1 of 4
// 20,000 pairs 23.7 | 22.6, top-2 of 16 16,000 19.8 | 19.4, 18,000 20.1 | 21.5, top-4 of 48 18,000 18.9 | 20.4, top-8 of 128 18,000 20.2 | 20.8,
// 24,500 20.9 | 22.0; tables, uniform (Zipf), top-2 of 24 18,000 23.0 | 23.1 (25.9 | 24.9), 20,000 23.4 | 23.9 (26.3 | 26.1), top-4 of 48
// 20,000 23.2 | 23.8 (25.3 | 25.2), 24,500 23.9 | 25.8 (26.4 | 27.4), top-8 of 128 24,500 25.9 | 25.5 (27.0 | 27.1).
static uint32_t sort_one_launch(const ItemSource &src) {
    if (src.n_experts > 128) return kSortRuns * kScanThreads;
    if (src.pairs) return src.n_experts > 4 ? 16384u : 20480u;
    return src.n_experts > 64 ? 24576u : 20480u;
}
// (256 threads up to 2,048 items: fewer waves to meet)
static uint32_t sort_threads(uint32_t n_items) { return n_items <= 2048 ? 256 : kScanThreads; }
__global__ __launch_bounds__(kScanThreads) void prefill_sort_kernel(ItemSource src, PrefillPlan *__restrict__ plan,
                                                                    PrefillTile *__restrict__ tiles, uint32_t max_tiles,
                                                                    TileRows bm, uint32_t *__restrict__ sorted_token,
                                                                    uint32_t *__restrict__ sorted_out_row) {
    __shared__ uint32_t cnt[FFMOE_MAX_EXPERTS], wave_own[kScanThreads / 64];
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6, mine = blockIdx.x;
    for (uint32_t c = threadIdx.x; c < FFMOE_MAX_EXPERTS; c += blockDim.x) cnt[c] = 0;
    __syncthreads();
    const uint32_t runs = (src.n_items + blockDim.x - 1) / blockDim.x, first = wave * runs * 64 + lane;
    unsigned long long own = 0ull;
    constexpr uint32_t kAhead = 8;
    for (uint32_t u0 = 0; u0 < runs; u0 += kAhead) {
        uint32_t e[kAhead];
        if (src.pairs) {
            uint32_t token[kAhead], rank[kAhead];
#pragma unroll
            for (uint32_t u = 0; u < kAhead; ++u) {
                const ffmoe_pair &p = src.pairs[min(first + (u0 + u) * 64, src.n_items - 1)];
                token[u] = p.token, e[u] = p.expert, rank[u] = p.rank;
            }
#pragma unroll
            for (uint32_t u = 0; u < kAhead; ++u) e[u] = ((token[u] < src.t) & (rank[u] < src.top_k)) ? e[u] : 0xFFFFFFFFu;
        } else {
            // zero-weight routes are dropped, as the reference's prefill does (RealForwardRunner.swift:1528-1530)
            uint16_t w[kAhead];
#pragma unroll
            for (uint32_t u = 0; u < kAhead; ++u) {
                const uint32_t i = min(first + (u0 + u) * 64, src.n_items - 1);
                e[u] = src.idx[i], w[u] = src.w[i];
            }
#pragma unroll
            for (uint32_t u = 0; u < kAhead; ++u) e[u] = (w[u] & 0x7FFFu) != 0 ? e[u] : 0xFFFFFFFFu;
        }
#pragma unroll
        for (uint32_t u = 0; u < kAhead; ++u) {
            const bool valid = u0 + u < runs && first + (u0 + u) * 64 < src.n_items && e[u] < src.n_experts;
            uint32_t same = 1;
            bool adds = valid;
            if (src.pairs) {
                // lists come sorted by expert: 64 lanes at one counter would take turns, so the first of a row of equals adds for all
                // (8,000 pairs in order: 14.7 -> 7.4 us; a table of top-1 routes, 20,480 random ones, would take 3 us more so)
                const uint32_t key = valid ? e[u] : 0xFFFFFFFFu, before = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)key, 0x138, 0xf, 0xf, false);    // (wave_shr:1)
                const unsigned long long heads = __ballot(lane == 0 || key != before) >> lane >> 1;
                adds = valid && (lane == 0 || key != before);
                same = heads ? (uint32_t)__builtin_ctzll(heads) + 1 : 64 - lane;
            }
            if (adds) atomicAdd(&cnt[e[u]], same);
            own |= (unsigned long long)(valid && e[u] == mine) << ((u0 + u) & 63);
        }
    }
    // (counts up to kSortRuns * kScanThreads: exact in fp32, as are the sums below)
    const uint32_t n_wave = (uint32_t)wave_butterfly_sum((float)__popcll(own));
    if (lane == 0) wave_own[wave] = n_wave;
    __syncthreads();
    uint32_t n[FFMOE_MAX_EXPERTS / 64];
    float in_front = 0.0f;
#pragma unroll
    for (uint32_t k = 0; k < FFMOE_MAX_EXPERTS / 64; ++k) {
        n[k] = cnt[64 * k + lane];                          // (experts past the last hold zero)
        if (64 * k + lane < mine) in_front += (float)n[k];
    }
    const uint32_t row0 = (uint32_t)wave_butterfly_sum(in_front);
    uint32_t pos = row0;
    for (uint32_t v = 0; v < wave; ++v) pos += wave_own[v];
    if (n_wave) {
        for (uint32_t u = 0; u < runs; ++u) {
            const unsigned long long with = __ballot((own >> u) & 1ull);
            if ((own >> u) & 1ull) place_item(src, first + u * 64, pos + (uint32_t)__popcll(with & ((1ull << lane) - 1ull)), sorted_token, sorted_out_row);
            pos += (uint32_t)__popcll(with);
        }
    }
    if (wave != waves - 1) return;
    // The tile list runs from the largest tile down: the full tiles in expert order, then every expert's last, shorter
    // tile by its rows (ties in expert order). The GEMM grids walk the list eight tiles at a time, so the launches end
    // with their shortest blocks instead of with whatever the last experts hold (a Zipf chunk's heavy experts sit
    // anywhere in the expert order).
    const uint32_t n_mine = cnt[mine], whole_mine = bm.whole(n_mine), rest_mine = n_mine - whole_mine * bm.rows;
    float full_front = 0.0f, full = 0.0f, pairs = 0.0f;
    uint32_t shorter_front = 0, shorter = 0, above = 0, with_pairs = 0;
#pragma unroll
    for (uint32_t k = 0; k < FFMOE_MAX_EXPERTS / 64; ++k) {
        const uint32_t o = 64 * k + lane, whole = bm.whole(n[k]), rest = n[k] - whole * bm.rows;
        const bool front = o < mine;
        full += (float)whole, pairs += (float)n[k];
        full_front += front ? (float)whole : 0.0f;
        with_pairs += (uint32_t)__popcll(__ballot(n[k] != 0));
        shorter += (uint32_t)__popcll(__ballot(rest != 0));
        shorter_front += (uint32_t)__popcll(__ballot(rest != 0 && front));
        above += (uint32_t)__popcll(__ballot(rest > rest_mine || (rest != 0 && rest == rest_mine && front)));
    }
    const uint32_t full_in_front = (uint32_t)wave_butterfly_sum(full_front), full_tiles = (uint32_t)wave_butterfly_sum(full);
    // a tile keeps its number in row order, which places its activation blocks
    for (uint32_t i = lane; i < whole_mine + (rest_mine != 0 ? 1u : 0u); i += 64) {
        const uint32_t ti = i < whole_mine ? full_in_front + i : full_tiles + above;
        if (ti < max_tiles) {
            PrefillTile tl;
            tl.expert = mine;
            tl.row_start = row0 + i * bm.rows;
            tl.rows = min(bm.rows, n_mine - i * bm.rows);
            tl.order = full_in_front + shorter_front + i;
            tiles[ti] = tl;
        }
    }
    const uint32_t n_pairs = (uint32_t)wave_butterfly_sum(pairs);
    if (lane != 0) return;
    plan->expert_offset[mine] = row0;
    plan->expert_count[mine] = n_mine;
    if (mine == 0) {
        plan->n_pairs = n_pairs;
        plan->n_tiles = min(full_tiles + shorter, max_tiles);
        plan->live_experts = with_pairs;
        plan->expert_offset[src.n_experts] = n_pairs;
    }
}

__global__ __launch_bounds__(kSortBlock) void prefill_scatter_kernel(ItemSource src, const uint32_t *__restrict__ block_base,
                                                                     uint32_t *__restrict__ sorted_token,
                                                                     uint32_t *__restrict__ sorted_out_row) {
    // an item's place inside its block's share of its expert = the items of the same expert in front of it: those in
    // the waves in front (per-wave counts in LDS) plus those in lower lanes of its own wave
    __shared__ uint32_t wave_cnt[kSortBlock / 64][FFMOE_MAX_EXPERTS];
    const uint32_t i = blockIdx.x * kSortBlock + threadIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (uint32_t c = threadIdx.x; c < (kSortBlock / 64) * FFMOE_MAX_EXPERTS; c += kSortBlock) (&wave_cnt[0][0])[c] = 0;
    const uint32_t e = item_expert(src, i);
    const bool valid = e != 0xFFFFFFFFu;
    const unsigned long long same = same_expert(e);
    const uint32_t in_front = __popcll(same & ((1ull << lane) - 1ull));
    __syncthreads();
    if (valid && in_front == 0) wave_cnt[wave][e] = __popcll(same);
    __syncthreads();
    if (!valid) return;
    uint32_t rank = in_front;
    for (uint32_t v = 0; v < wave; ++v) rank += wave_cnt[v][e];
    place_item(src, i, block_base[(size_t)blockIdx.x * src.n_experts + e] + rank, sorted_token, sorted_out_row);
}

// A dense FFN's chunk needs no sort: one expert, route r = row r. One launch writes what the three above would: the
// identity tables and the chunk cut into M-tiles.
__global__ __launch_bounds__(kSortBlock) void prefill_dense_plan_kernel(uint32_t t, uint32_t bm,
                                                                       PrefillPlan *__restrict__ plan,
                                                                       PrefillTile *__restrict__ tiles,
                                                                       uint32_t *__restrict__ sorted_token,
                                                                       uint32_t *__restrict__ sorted_out_row) {
    const uint32_t i = blockIdx.x * kSortBlock + threadIdx.x;
    if (i < t) {
        sorted_token[i] = i;
        sorted_out_row[i] = i;
    }
    const uint32_t n_tiles = (t + bm - 1) / bm;          // bm: a multiple of 16, at most kBM
    if (i < n_tiles) {
        PrefillTile tl;
        tl.expert = 0;
        tl.row_start = i * bm;
        tl.rows = min(bm, t - i * bm);
        tl.order = i;
        tiles[i] = tl;
    }
    if (i == 0) {
        plan->n_pairs = t;
        plan->n_tiles = n_tiles;
        plan->live_experts = 1;
        plan->expert_count[0] = t;
        plan->expert_offset[0] = 0;
        plan->expert_offset[1] = t;
    }
}

// ---------------------------------------------------------------------------------------------------
// Grouped GEMM. One block = one M-tile (up to 256 pairs of one expert) x one N-block (8 arena tiles = 256 weight rows), a wave
// per arena tile: its 32 weight rows against all pairs of the tile.
//   Weights: a lane's 16 bytes of an arena tile are its share of four matrix operands already, so they are expanded to
//      bf16(fma(q, scale, bias)) register to register, an operand set ahead of the products, once per M-tile; the packed tiles go
//      from memory straight into LDS, kRingW groups ahead.
//   Pairs: a 64-wide group of their rows goes from memory straight into LDS as well (three buffers), and every wave reads each
//      16-pair fragment once and multiplies it with its two row blocks.
// A block of eight waves per compute unit, or two where tiles have up to 128 pairs (GemmLds), walks a list of such items
// (prefill_gemm_kernel), the loads running on from one to the next.
// What bounds it: 192 pairs per expert make 48 matrix instructions per wave and group, i.e. 1,536 cycles of a SIMD's matrix unit
// of the 2,150 that a group takes; beside them 82 vector instructions (the expansion, 68 of them, shrinks with every pair a
// wave multiplies its weights with), 26 LDS reads and one barrier. Run back to back the card also lowers its clock under it.
// Weights through LDS instead (a wave expands a tile for all waves to read) costs the same however the waves split a block:
// 215 to 235 us where this takes 183; 64 weight rows x 128 pairs per wave, every tile expanded twice, 209. Gate/up and down of a
// 3,072-row chunk 222 + 115 -> 183 + 110 us, of 8,192 skewed rows 7.5 % less per layer, of 1,000 FP16 rows 144 + 78 -> 114 + 68 (102 + 59 with two blocks per unit); 256 pairs in each of 128
// experts 275 + 133 -> 216 + 137 us (1,200 TFLOP/s in gate/up). A second pass of bf16 products by the vendor's library on ready-made
// weights reaches 1,250 on this card.
// GATE_UP: A rows are gathered token rows of x; streams are gate / up; out = the activations, stored in the order the
//          down GEMM's matrix instructions want them (below).
// else:    A = those activations; streams are two 16-row blocks; out = partials[out_row][D] (16-bit).
// Activation layout: [16-pair block][group of F][k-half][lane (j, jq)] x 8 values = pair j of the block at
// k = 32 * (k-half) + 8 * jq .. + 7 of the group. The 16-pair blocks of an M-tile start at block row_start / 16 + its number
// in row order: consecutive tiles never share a block (a tile adds at most one block of slack), so the buffer holds
// max_pairs / 16 + max_tiles + 1 blocks.
// ---------------------------------------------------------------------------------------------------

struct GemmWave {
    const uint16_t *a;                    // A matrix
    uint32_t a_stride, n_groups, n_arena_tiles, nb, wave, lane;
    uint32_t act_blocks;                  // 16-pair blocks the activation buffer holds (the scale tables' extent)
    uint32_t act_block0;                  // first 16-pair block of this M-tile in the activation layout
    PrefillTile tile;
};

constexpr int kGemmTiles = 8;                               // arena tiles per N-block = waves per block
constexpr uint32_t kFragBytes = kWave * 16;                 // one matrix operand of a wave
constexpr uint32_t kGemmWBytes = kTileBytes + 2 * kTileScaleBytes;            // packed tile of one wave (a 64-lane load brings the scales twice)
constexpr uint32_t kGemmTurnRow = 2 * kTileRows * 2 + 16, kGemmTurnBytes = 16 * kGemmTurnRow;
// A block whose tiles have up to 64 LC pairs. Tiles of up to 128 leave registers (128 per wave) and LDS for two such blocks per compute
// unit: four waves per SIMD have more to issue while one waits for the matrix unit, LDS or a barrier. Gate/up and down of 1,000 rows,
// 62 pairs per expert, 99 + 62 us with one block | 89 + 51 with two; a wave then is picked for an instruction in 87 % of its SIMD's issue
// slots, 77 % before. Beyond 128 pairs a wave's sums take the registers of two.
template <int LC>
struct GemmLds {
    static constexpr int kBlocks = LC == 2 ? 2 : 1;                     // of a compute unit
    static constexpr int kRingA = 3, kRingW = LC == 2 ? 3 : 5;          // groups of A, and of packed tiles at most
    static constexpr uint32_t kABytes = 4 * LC * 2 * kFragBytes;
    static constexpr uint32_t kWAt = kRingA * kABytes, kRowAt = kWAt + kRingW * kGemmTiles * kGemmWBytes;
    // (down product: the pairs' output rows and largest scales, two items' worth)
    static constexpr uint32_t kRowBytes = 64 * LC * 4, kLargestAt = kRowAt + 2 * kRowBytes;
    // the epilogues work in the buffer of the item's last group of A: the next item's first two are in the others
    static constexpr int kTurnBlocks = LC == 2 ? 1 : 3;                 // 16-pair blocks that a wave turns at a time
    static constexpr uint32_t bytes(bool gate_up, bool f16) { return gate_up ? kRowAt : f16 ? kLargestAt + 2 * kRowBytes : kLargestAt; }
    static_assert(kGemmTiles * kTurnBlocks * kGemmTurnBytes <= kABytes && kGemmTiles * 64 * LC * 4 <= kABytes, "staging rows or peaks fit a buffer");
    static_assert(kBlocks * (kLargestAt + 2 * kRowBytes) <= 160 * 1024, "a compute unit's LDS");
};

// One M-tile x N-block, and what a wave needs to ask for its rows: `from` = GATE_UP: in bytes from the first row's start (WIDE, where
// the rows span 4 GiB or more: the row); else: in KiB, wave-uniform.
template <int LC>
struct GemmItem {
    bool valid;
    uint32_t parity;                      // of its number among the block's
    PrefillTile tile;
    uint32_t nb, act_block0, loads;
    uint32_t from[LC];
    const uint8_t *w_tiles, *w_scales;    // this wave's arena tile
};

// How many fragments of A a wave has in flight or in use, `most` or fewer: a divisor of the 2 NM of a group, so that a fragment's
// registers are known at compile time, and at most NM + 1, so that none of the next group is read in a group's first half.
constexpr int gemm_queue(int nm, int most) {
    if ((nm == 11 || nm == 13) && most > 4) return nm;
    int q = 2;
    for (int d = 3; d <= most; ++d)
        if (2 * nm % d == 0 && d <= nm + 1) q = d;
    return q;
}

// NM: 16-pair blocks of the tile, all of them this wave's (a compile-time count: the matrix instructions have no branches
// between them); 0 for a wave past the last arena tile, which only brings its share of A. LOADS: KiB of A per wave and group.
// DUMP: a test instantiation that also copies every weight operand out, so that a test can hold the expanded tile itself
// against the reference's 16-bit weight.
// F16: the reference's FP16 prefill (prefill.metal:581-598,685-702,723-777): FP16 rows against FP16 tile weights
// half(fma(q, scale, bias)), fp32 sums; the activations between the two GEMMs are FP16 with a power-of-two scale per
// pair and 64-wide block of F (`act_scale[pair][block]`; the block's largest magnitude lands below 2^14), so values
// past FP16's range keep FP16's relative precision; a pass between the two brings every block of a pair to the pair's largest
// scale (exact unless a value falls below FP16's normal range relative to that largest) and the down GEMM applies that scale
// to the pair's sums.
// Where a wave is in the rings, as byte offsets into LDS: they turn on from one item to the next.
struct GemmRings {
    uint32_t cur, next, before;           // A of the group at hand, of the next one, of the one before (and of the group after the next)
    uint32_t slot, first_slot, end_slot;  // this wave's packed tile of the group at hand; where its slots begin and end
    uint32_t depth;                       // slots in use
    __device__ __forceinline__ uint32_t next_slot() const {
        const uint32_t s = slot + kGemmTiles * kGemmWBytes;
        return s == end_slot ? first_slot : s;
    }
    __device__ __forceinline__ void turn() {
        const uint32_t c = cur;
        cur = next, next = before, before = c;
        slot = next_slot();
    }
};

// The 16-byte piece of its row's 128 bytes that a lane brings.
__device__ __forceinline__ uint32_t gemm_row_piece(uint32_t lane) { return (lane & 7) ^ (lane >> 3); }
// The loads of one group: the k-th KiB of a wave's share of A, its packed tile (k = 0) and that tile's scales (k = 1).
template <bool GATE_UP, bool F16, bool WIDE, int LC>
__device__ __forceinline__ void gemm_load_a(const GemmWave &gw, const GemmItem<LC> &it, uint32_t lds_base, uint32_t grp, uint32_t at, int k) {
    const uint32_t to = lds_base + at + (gw.wave + kGemmTiles * k) * kFragBytes;
    if constexpr (GATE_UP && WIDE) global_to_lds_16(gw.a + grp * kGroup + (size_t)it.from[k] * gw.a_stride + gemm_row_piece(gw.lane) * 8, to);
    else if constexpr (GATE_UP) global_to_lds_16(gw.a + grp * kGroup, it.from[k], to);
    else global_to_lds_16(gw.a + ((size_t)it.from[k] + 2 * grp) * (kWave * 8), gw.lane * 16, to);
}
__device__ __forceinline__ void gemm_load_w(uint32_t lane, const uint8_t *w_tiles, const uint8_t *w_scales, uint32_t to, int k) {
    if (k == 0) global_to_lds_16(w_tiles, lane * 16, to);
    else global_to_lds_4(w_scales, lane * 4 % kTileScaleBytes, to + kTileBytes);
}
// what an item's first step counts on: two groups of A, as many packed tiles as the ring holds
template <bool GATE_UP, bool F16, bool WIDE, int LC>
__device__ __forceinline__ void gemm_ask(const GemmWave &gw, const GemmItem<LC> &it, uint32_t lds_base, const GemmRings &rings) {
#pragma unroll
    for (uint32_t grp = 0; grp < (uint32_t)GemmLds<LC>::kRingW; ++grp) {
        const bool live = grp < rings.depth;
        const uint32_t to = lds_base + rings.first_slot + grp * kGemmTiles * kGemmWBytes;
        if (live) {
            gemm_load_w(gw.lane, it.w_tiles + grp * kTileBytes, it.w_scales + grp * kTileScaleBytes, to, 0);
            gemm_load_w(gw.lane, it.w_tiles + grp * kTileBytes, it.w_scales + grp * kTileScaleBytes, to, 1);
        }
        if (grp < 2 && live) {
#pragma unroll
            for (int k = 0; k < LC; ++k)
                if ((uint32_t)k < it.loads)
                    gemm_load_a<GATE_UP, F16, WIDE>(gw, it, lds_base, grp, grp ? rings.next : rings.cur, k);
        }
    }
}

// What an item leaves. Nobody reads the last group of A any more; `stage` is its buffer.
template <bool GATE_UP, int NM, bool F16, bool DUMP, int LC>
__device__ __forceinline__ void gemm_epilogue(const GemmWave &gw, const GemmItem<LC> &it, const ArenaGeom &g, const uint8_t *lds, uint8_t *stage, uint32_t tile,
                                              uint32_t lane, f32x4 (&acc)[NM > 0 ? NM : 1][2], uint16_t *__restrict__ out, float *__restrict__ act_scale) {
    using L = GemmLds<LC>;
    constexpr int NA = NM > 0 ? NM : 1;
    const uint32_t wave = gw.wave, j = lane & 15, jq = lane >> 4;
    // lane (j, jq) holds pair j of every 16-pair block, weight rows 4 jq .. 4 jq + 3 of both row blocks
    if constexpr (GATE_UP) {
        // this wave's arena tile is k = 16 (tile % 4) .. + 15 of group tile / 4 of F: k-half tile / 2 % 2, operand lane
        // (j, 2 (tile % 2) + jq / 2), values 4 (jq % 2) .. + 3 of that lane's eight
#pragma unroll
        for (int i = 0; i < NA; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][0][r] = gelu_tanh_fast(acc[i][0][r]) * acc[i][1][r];
        if constexpr (F16) {
            // a pair's 64 activations of a group sit in the four lanes (j, 0..3) of four waves: their largest magnitude
            // peak < 2^e goes to 2^14 (frexp / ldexp as prefill.metal:689-702)
            float *peaks = reinterpret_cast<float *>(stage);                // [wave][pair]
#pragma unroll
            for (int i = 0; i < NM; ++i) {
                float peak = 0.0f;
#pragma unroll
                for (int r = 0; r < 4; ++r) peak = fmaxf(peak, fabsf(acc[i][0][r]));
                peak = fmaxf(peak, __shfl_xor(peak, 16, 64));
                peak = fmaxf(peak, __shfl_xor(peak, 32, 64));
                if (jq == 0) peaks[wave * (16 * NM) + 16 * i + j] = peak;
            }
            lds_barrier();
#pragma unroll
            for (int i = 0; i < NM; ++i) {
                float peak = 0.0f;
#pragma unroll
                for (uint32_t v = 0; v < 4; ++v) peak = fmaxf(peak, peaks[((wave & 4) + v) * (16 * NM) + 16 * i + j]);
                int e = 0;
                (void)frexpf(peak, &e);
                e = max(e, -100);                                   // 2^(14 - e) stays finite for a block of denormal size
                const float to_half = ldexpf(1.0f, 14 - e);
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[i][0][r] *= to_half;
                if (jq == 0 && (wave & 3) == 0 && 16 * i + j < it.tile.rows)
                    act_scale[((size_t)(it.act_block0 + i) * g.gf + tile / kTilesPerBlock) * 16 + j] = ldexpf(1.0f, e - 14);
            }
        }
#pragma unroll
        for (int i = 0; i < NM; ++i) {
            if (16 * i + j >= it.tile.rows) continue;
            uint16_t *oblk = out + (((size_t)(it.act_block0 + i) * g.gf + tile / kTilesPerBlock) * 2 + (tile >> 1 & 1)) * (kWave * 8);
            *reinterpret_cast<uint2 *>(oblk + (((tile & 1) * 2 + (jq >> 1)) * 16 + j) * 8 + (jq & 1) * 4) =
                make_uint2(Act<F16>::pack(acc[i][0][0], acc[i][0][1]), Act<F16>::pack(acc[i][0][2], acc[i][0][3]));
        }
        return;
    }
    // Down projection: a 16-pair block of this wave's columns is 16 rows x 64 B. Each wave turns its blocks through a private piece
    // of LDS, so that four lanes store 64 contiguous bytes of a row, instead of 8-byte pieces 32 B apart per instruction.
    uint8_t *turn = stage + wave * (L::kTurnBlocks * kGemmTurnBytes);
    const uint32_t row = lane >> 2, chunk = lane & 3;                           // read side
#pragma unroll
    for (int i0 = 0; i0 < NM; i0 += L::kTurnBlocks) {
#pragma unroll
        for (int i = i0; i < i0 + L::kTurnBlocks && i < NM; ++i) {
            float pair_largest = 1.0f;
            if constexpr (F16) pair_largest = *reinterpret_cast<const float *>(lds + L::kLargestAt + it.parity * L::kRowBytes + (16 * i + j) * 4);
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                f32x4 v = acc[i][st];
                if constexpr (F16) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] *= pair_largest;         // the pair's sums back to their scale
                }
                *reinterpret_cast<uint2 *>(turn + (i - i0) * kGemmTurnBytes + j * kGemmTurnRow + st * 32 + 8 * jq) =
                    make_uint2(Act<F16>::pack(v[0], v[1]), Act<F16>::pack(v[2], v[3]));
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        uint4 v[L::kTurnBlocks];
        uint32_t orow[L::kTurnBlocks];
#pragma unroll
        for (int i = i0; i < i0 + L::kTurnBlocks && i < NM; ++i) {
            v[i - i0] = *reinterpret_cast<const uint4 *>(turn + (i - i0) * kGemmTurnBytes + row * kGemmTurnRow + 16 * chunk);
            orow[i - i0] = *reinterpret_cast<const uint32_t *>(lds + L::kRowAt + it.parity * L::kRowBytes + (16 * i + row) * 4);
        }
#pragma unroll
        for (int i = i0; i < i0 + L::kTurnBlocks && i < NM; ++i)
            if (16 * i + row < it.tile.rows && (!DUMP || tile < gw.n_arena_tiles)) *reinterpret_cast<uint4 *>(out + (size_t)orow[i - i0] * g.d + tile * (2 * kTileRows) + 8 * chunk) = v[i - i0];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// (lds is not __restrict__: the loads write the same memory through lds_base)
template <bool GATE_UP, int NM, int LOADS, bool F16, bool WIDE, bool DUMP, int LC>
__device__ __forceinline__ void gemm_wave(const GemmWave &gw, const GemmItem<LC> &it, const GemmItem<LC> &next_item, GemmRings &rings, const ArenaGeom &g,
                                          uint8_t *lds, uint32_t lds_base, const uint32_t *__restrict__ sorted_out_row,
                                          uint16_t *__restrict__ out, float *__restrict__ act_scale, uint4 *__restrict__ dump = nullptr) {
    using L = GemmLds<LC>;
    constexpr int NA = NM > 0 ? NM : 1;
    constexpr int kQueue = gemm_queue(NA, L::kBlocks == 1 ? 8 : WIDE && NM > 6 ? 2 : 4);
    // (the lane's number is taken anew here and for the epilogue: what the compiler derives from it for every tile height it would
    // otherwise compute in front of the list of items and keep in scratch memory)
    uint32_t lane = gw.lane;
    asm volatile("" : "+v"(lane));
    const uint32_t wave = gw.wave, j = lane & 15, jq = lane >> 4, n_groups = gw.n_groups;
    const uint32_t tile = it.nb * kGemmTiles + wave;        // this wave's arena tile
    if constexpr (!GATE_UP) {
        // the pairs' output rows (and largest scales), for the epilogue; waves LC.. repeat what waves 0..LC - 1 bring
        const uint32_t pair = min((wave % LC) * kWave + lane, it.tile.rows - 1);
        global_to_lds_4(sorted_out_row + it.tile.row_start + pair, lds_base + L::kRowAt + it.parity * L::kRowBytes + (wave % LC) * (kWave * 4));
        if constexpr (F16)
            global_to_lds_4(act_scale + (size_t)gw.act_blocks * g.gf * 16 + it.act_block0 * 16 + pair, lds_base + L::kLargestAt + it.parity * L::kRowBytes + (wave % LC) * (kWave * 4));
    }
    uint4 wraw = {0, 0, 0, 0};
    uint2 sraw = {0, 0};
    auto read_w = [&](uint32_t slot) __attribute__((always_inline)) {
        const uint8_t *at = lds + slot;
        wraw = *reinterpret_cast<const uint4 *>(at + lane * 16);
        sraw = *reinterpret_cast<const uint2 *>(at + kTileBytes + j * 8);
    };
    // Expansion: bits 0..3 and 4..7 of each half of a dword are FP16 subnormals q 2^-24 and q 2^-20 as they lie, and one
    // v_fma_mix_f32 takes such a half with fp32 scale (times 2^24, 2^20: exact below 2^104, and layers with larger ones do not come
    // here) and bias: 17 vector instructions for eight weights instead of 23 with byte conversions, the same fp32 value to the bit.
    float s24[2], s20[2], bias[2];
    auto take_scales = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            const uint32_t sb = st ? sraw.y : sraw.x;
            s24[st] = bf16lo_to_f32(sb) * 16777216.0f;
            s20[st] = bf16lo_to_f32(sb) * 1048576.0f;
            bias[st] = bf16hi_to_f32(sb);
        }
    };
    uint4 wf[2][2];                     // operands: k-half, stream
    auto expand_piece = [&](int half, int piece) __attribute__((always_inline)) {
        // half of a dword: two packed pairs at a time, so that the conversion of one stands behind the products of the other
        const int st = piece >> 1;
        const uint32_t w = st ? (half ? wraw.w : wraw.z) : (half ? wraw.y : wraw.x), b = piece & 1 ? w >> 8 : w;
        const f16x2 u = __builtin_bit_cast(f16x2, b & 0x000F000Fu), v = __builtin_bit_cast(f16x2, b & 0x00F000F0u);
        const float u0 = __builtin_fmaf((float)u[0], s24[st], bias[st]), u1 = __builtin_fmaf((float)u[1], s24[st], bias[st]);
        const float v0 = __builtin_fmaf((float)v[0], s20[st], bias[st]), v1 = __builtin_fmaf((float)v[1], s20[st], bias[st]);
        uint32_t lo = Act<F16>::pack(u0, u1), hi = Act<F16>::pack(v0, v1);
        asm volatile("" : "+v"(lo), "+v"(hi));     // here, among the products, and not where the operand is first used
        if (piece & 1) wf[half][st].z = lo, wf[half][st].w = hi;
        else wf[half][st].x = lo, wf[half][st].y = hi;
    };

    f32x4 acc[NA][2];
#pragma unroll
    for (int i = 0; i < NA; ++i) acc[i][0] = acc[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint4 xq[kQueue];
    // fragment f (k-half f / NM of 16-pair block f % NM) of a group
    const uint32_t at0 = GATE_UP ? j * 128 + 16 * (jq ^ (j & 7)) : lane * 16;
    auto read_a = [&](uint32_t from, int f) __attribute__((always_inline)) {
        const int half = f / NA, i = f % NA;
        const uint32_t at = GATE_UP ? at0 ^ (64 * half) : at0 + half * kFragBytes;
        xq[f % kQueue] = *reinterpret_cast<const uint4 *>(lds + from + i * (2 * kFragBytes) + at);
    };
    // One step = one group, its k-halves one after the other: the products with the four pieces of the next operand set's
    // expansion between them (a scheduling fence behind each product keeps them there) and the fragments of A kQueue - 1 ahead.
    // In its middle the next group's A, asked for in the step before, has to be there, and a barrier makes it the whole block's; the
    // last fragments' reads then run ahead into that group, and the buffer of the group before is filled again.
    // What a step asks for goes out between its products: all at once, the waves queue for the address unit (11 ns per KiB of
    // rows) in front of their products. Behind an item's last group comes the next item's first, so that its packed tiles and, in
    // the last two steps, its A are on their way before this one ends; without a next item this one's once more. (The last two steps
    // ask for a whole tile's rows, whatever the items have: behind a branch the compiler moves a step's products, and keeps all their
    // operands until there.)
    GemmItem<LC> next = it;
    if (next_item.valid) next = next_item;
    const uint8_t *const next_w_tiles = next.w_tiles, *const next_w_scales = next.w_scales;
    uint32_t own_w = n_groups - rings.depth;                        // groups of this item whose packed tiles are still to be asked for
    const uint8_t *ask_tiles = own_w ? it.w_tiles + rings.depth * kTileBytes : next_w_tiles;
    const uint8_t *ask_scales = own_w ? it.w_scales + rings.depth * kTileScaleBytes : next_w_scales;
    auto step = [&](uint32_t grp, auto is_steady) __attribute__((always_inline)) {
        constexpr bool kSteady = decltype(is_steady)::value;        // not one of the last two: A is this item's, and no branches
        constexpr int kUnits = 2 * NA;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            if (half == 1) {
                if (DUMP) vmem_barrier<0>();
                else vmem_barrier<2>();                             // (the packed tile asked for in the first half)
                if (NM > 0) read_w(rings.next_slot());
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (DUMP && NM > 0) {
#pragma unroll
                for (int st = 0; st < 2; ++st)
                    dump[(((size_t)(tile / kTilesPerBlock) * n_groups + grp) * 16 + half * 8 + tile % kTilesPerBlock * 2 + st) * kWave + lane] = wf[half][st];
            }
            constexpr int kFirst = NA > 2 ? 4 : 0;
            const int first = half == 1 ? kFirst : 0;               // (the packed tile is on its way from LDS)
#pragma unroll
            for (int i = 0; i < NA; ++i) {
                const int f = half * NM + i, ahead = f + kQueue - 1;
                uint4 x = {0, 0, 0, 0};
                if (NM > 0) {
                    if (ahead < 2 * NM) read_a(rings.cur, ahead);
                    else read_a(rings.next, ahead - 2 * NM);
                    x = xq[f % kQueue];
                }
#pragma unroll
                for (int st = 0; st < 2; ++st) {
                    // weights as the first operand: the lane ends up with four consecutive weight rows of
                    // one pair, which the epilogue packs into one 8-byte piece of that pair's output row
                    if (NM > 0) acc[i][st] = Act<F16>::mfma(wf[half][st], x, acc[i][st]);
                    const int at = 2 * i + st, u = at - first;
                    if (half == 1 && kSteady) {
#pragma unroll
                        for (int k = 0; k < LOADS; ++k)
                            if (at == max((k + 1) * kUnits / (LOADS + 1) - 1, 0)) gemm_load_a<GATE_UP, F16, WIDE>(gw, it, lds_base, grp + 2, rings.before, k);
                    } else if (half == 1) {
#pragma unroll
                        for (int k = 0; k < LC; ++k)
                            if (at == max((k + 1) * kUnits / (LC + 1) - 1, 0))
                                gemm_load_a<GATE_UP, F16, WIDE>(gw, next, lds_base, min(grp + 2 - n_groups, n_groups - 1), rings.before, k);
                    } else {
#pragma unroll
                        for (int k = 0; k < 2; ++k)
                            if (at == max((k + 1) * kUnits / 3 - 1, 0))      // (this group's went to registers in the step before)
                                gemm_load_w(lane, ask_tiles, ask_scales, lds_base + rings.slot, k);
                    }
                    if (NM > 0) {
                        if (half == 1 && u == 0) take_scales();
#pragma unroll
                        for (int p = max(u, 0) * 4 / (kUnits - first); p < max(u + 1, 0) * 4 / (kUnits - first); ++p) expand_piece(half ^ 1, p);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    };
    if (NM > 0) {
        read_w(rings.slot);
        take_scales();
#pragma unroll
        for (int p = 0; p < 4; ++p) expand_piece(0, p);
#pragma unroll
        for (int f = 0; f < kQueue - 1; ++f) read_a(rings.cur, f);
    }
    auto turn_rings = [&]() __attribute__((always_inline)) {
        rings.turn();
        ask_tiles += kTileBytes;
        ask_scales += kTileScaleBytes;
        if (--own_w == 0) ask_tiles = next_w_tiles, ask_scales = next_w_scales;
    };
    uint32_t grp = 0;
#pragma nounroll
    for (; grp + 2 < n_groups; ++grp) {
        step(grp, std::true_type{});
        turn_rings();
    }
#pragma nounroll
    for (; grp < n_groups; ++grp) {
        step(grp, std::false_type{});
        turn_rings();
    }
    lds_barrier();                      // nobody reads the last group's A any more
    uint8_t *const stage = lds + rings.before;
    if (n_groups == 1 && next_item.valid) gemm_ask<GATE_UP, F16, WIDE>(gw, next_item, lds_base, rings);

    uint32_t out_lane = gw.lane;
    asm volatile("" : "+v"(out_lane));
    gemm_epilogue<GATE_UP, NM, F16, DUMP, LC>(gw, it, g, lds, stage, tile, out_lane, acc, out, act_scale);
}

// Consecutive block ids go to consecutive XCDs. Many experts: all N-blocks of an M-tile share an XCD (its L2 holds
// the tile's A rows). One expert (the dense FFN: few M-tiles, every one against the same weights): all M-tiles of
// an N-block share an XCD instead, so each XCD reads its eighth of the weights once and every XCD is equally full.
__device__ __forceinline__ bool prefill_block(uint32_t n_nblocks, bool nb_major, uint32_t &tile, uint32_t &nb) {
    const uint32_t xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    if (nb_major) {
        const uint32_t per_xcd = (n_nblocks + 7) / 8;
        tile = slot / per_xcd;
        nb = (slot % per_xcd) * 8 + xcd;
        return nb < n_nblocks;
    }
    tile = (slot / n_nblocks) * 8 + xcd;
    nb = slot % n_nblocks;
    return true;
}

// F16: a context in FP16 mode - FP16 rows in, FP16 tiles, block-scaled FP16 activations, FP16 per-route rows out.
// A block works off its share of the XCD's items one after the other: an item's first loads then travel
// during the epilogue of the one before.
template <bool GATE_UP, bool F16, bool WIDE, int LC, bool DUMP = false>
__global__ __launch_bounds__(64 * kGemmTiles, 2 * GemmLds<LC>::kBlocks) void prefill_gemm_kernel(const uint8_t *__restrict__ arena_layer, ArenaGeom g,
                                                                          const PrefillPlan *__restrict__ plan,
                                                                          const PrefillTile *__restrict__ tiles,
                                                                          const uint32_t *__restrict__ sorted_token,
                                                                          const uint32_t *__restrict__ sorted_out_row,
                                                                          const uint16_t *__restrict__ a, uint32_t a_stride,
                                                                          uint16_t *__restrict__ out, bool nb_major,
                                                                          float *__restrict__ act_scale, uint32_t act_blocks,
                                                                          uint4 *__restrict__ dump = nullptr) {
    using L = GemmLds<LC>;
    __shared__ __align__(16) uint8_t lds[L::bytes(GATE_UP, F16)];
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
    GemmWave gw;
    gw.lane = threadIdx.x & 63;
    gw.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);      // wave-uniform: branches on it stay scalar
    gw.n_groups = GATE_UP ? g.gd : g.gf;
    gw.n_arena_tiles = GATE_UP ? g.gu_rb : g.dn_rbp;
    gw.a = a;
    gw.a_stride = a_stride;
    gw.act_blocks = act_blocks;

    // The XCD's items, largest first: full N-blocks tile by tile, then the tiles' last N-blocks where those are not full, then its
    // share of the tiles that do not make up a set of eight.
    // Many experts: an M-tile's items are all on one XCD (its L2 holds the tile's A rows), tile t on XCD t % 8, but for the last few. One
    // expert (the dense FFN: few M-tiles, every one against the same weights): the N-blocks one after the other, an eighth of the
    // list per XCD, so that each reads its eighth of the weights once.
    const uint32_t xcd = blockIdx.x & 7, mine = blockIdx.x >> 3, per_xcd = gridDim.x >> 3;
    const uint32_t n_tiles = plan->n_tiles, n_full = gw.n_arena_tiles / kGemmTiles, n_nb = (gw.n_arena_tiles + kGemmTiles - 1) / kGemmTiles;
    const uint32_t all = n_tiles * n_nb, tiles_x = n_tiles / 8, over = n_tiles % 8 * n_nb;
    const uint32_t first = nb_major ? (uint32_t)((uint64_t)all * xcd / 8) : 0;
    const uint32_t n_items = nb_major ? (uint32_t)((uint64_t)all * (xcd + 1) / 8) - first : tiles_x * n_nb + (over + 7 - xcd) / 8;
    // round r of this block: the rounds run forth and back over the blocks, so that who had a large item gets a small one
    auto item_at = [&](uint32_t r) __attribute__((always_inline)) {
        GemmItem<LC> it;
        const uint32_t q = r * per_xcd + (r & 1 ? per_xcd - 1 - mine : mine);
        it.valid = q < n_items;
        it.parity = r & 1;
        if (!it.valid) return it;
        uint32_t ti;
        if (nb_major) {
            ti = (first + q) % n_tiles;
            it.nb = (first + q) / n_tiles;
        } else if (q < tiles_x * n_full) {
            ti = q / n_full * 8 + xcd;
            it.nb = q % n_full;
        } else if (q < tiles_x * n_nb) {
            ti = (q - tiles_x * n_full) * 8 + xcd;
            it.nb = n_full;
        } else {
            const uint32_t o = (q - tiles_x * n_nb) * 8 + xcd;
            ti = tiles_x * 8 + o / n_nb;
            it.nb = o % n_nb;
        }
        ti = __builtin_amdgcn_readfirstlane(ti);
        it.nb = __builtin_amdgcn_readfirstlane(it.nb);
        it.tile = tiles[ti];
        it.tile.rows = __builtin_amdgcn_readfirstlane(it.tile.rows);
        it.act_block0 = it.tile.row_start / 16 + it.tile.order;
        const uint32_t last_block = (it.tile.rows - 1) / 16;
        it.loads = last_block / 4 + 1;
        // A to LDS, 1 KiB at a time. GATE_UP: eight rows of 128 bytes, eight neighbouring lanes per row; 16-byte piece c of row r lies
        // at piece c ^ (r % 8) of the row, so that the sixteen rows of a fragment read fall on different banks. else: the
        // activations are stored fragment by fragment.
#pragma unroll
        for (int k = 0; k < LC; ++k) {
            const uint32_t piece = gw.wave + kGemmTiles * k;
            if constexpr (GATE_UP) {
                const uint32_t row = min(piece * 8 + (gw.lane >> 3), it.tile.rows - 1);
                const uint32_t token = sorted_token[it.tile.row_start + row];
                it.from[k] = WIDE ? token : (token * (gw.a_stride / 8) + gemm_row_piece(gw.lane)) * 16u;
            } else {
                it.from[k] = __builtin_amdgcn_readfirstlane((it.act_block0 + min(piece >> 1, last_block)) * gw.n_groups * 2 + (piece & 1));
            }
        }
        // this wave's arena tile; past the last one the last again (read and left at that)
        const uint32_t at = min(it.nb * kGemmTiles + gw.wave, gw.n_arena_tiles - 1) * gw.n_groups;
        const uint8_t *expert_base = arena_layer + (size_t)__builtin_amdgcn_readfirstlane(it.tile.expert) * g.expert_bytes;
        it.w_tiles = expert_base + (GATE_UP ? g.gu_tiles_off : g.dn_tiles_off) + (size_t)at * kTileBytes;
        it.w_scales = expert_base + (GATE_UP ? g.gu_scales_off : g.dn_scales_off) + (size_t)at * kTileScaleBytes;
        return it;
    };
    GemmItem<LC> it = item_at(0);
    if (!it.valid) return;
    GemmRings rings;
    rings.depth = min((uint32_t)L::kRingW, gw.n_groups);
    rings.cur = 0, rings.next = L::kABytes, rings.before = 2 * L::kABytes;
    rings.slot = rings.first_slot = L::kWAt + gw.wave * kGemmWBytes;
    rings.end_slot = rings.first_slot + rings.depth * (kGemmTiles * kGemmWBytes);
    gemm_ask<GATE_UP, F16, WIDE>(gw, it, lds_base, rings);
    vmem_barrier<0>();
    for (uint32_t r = 1;; ++r) {
        const GemmItem<LC> next = item_at(r);
        const uint32_t n_mb = (it.tile.rows + 15) / 16;
        // (the test's tiles past the last, up to a set of four, are the last once more)
        const uint32_t owned = DUMP ? (gw.n_arena_tiles + kTilesPerBlock - 1) / kTilesPerBlock * kTilesPerBlock : gw.n_arena_tiles;
        const bool owns = it.nb * kGemmTiles + gw.wave < owned;
        // (waves that own no tile take part in the loads and the barriers, which are the same in all instantiations of one LOADS)
#define FFMOE_GEMM_WAVE(N, K) if constexpr (K <= LC) gemm_wave<GATE_UP, N, K, F16, WIDE, DUMP, LC>(gw, it, next, rings, g, lds, lds_base, sorted_out_row, out, act_scale, dump)
        if constexpr (DUMP) {
            // the test launch runs one pair
            if (owns) { FFMOE_GEMM_WAVE(1, 1); } else { FFMOE_GEMM_WAVE(0, 1); }
        } else if (!owns) {
            switch ((n_mb + 3) / 4) {
                case 1: FFMOE_GEMM_WAVE(0, 1); break;
                case 2: FFMOE_GEMM_WAVE(0, 2); break;
                case 3: FFMOE_GEMM_WAVE(0, 3); break;
                default: FFMOE_GEMM_WAVE(0, 4); break;
            }
        } else {
            switch (n_mb) {
                case 1: FFMOE_GEMM_WAVE(1, 1); break;
                case 2: FFMOE_GEMM_WAVE(2, 1); break;
                case 3: FFMOE_GEMM_WAVE(3, 1); break;
                case 4: FFMOE_GEMM_WAVE(4, 1); break;
                case 5: FFMOE_GEMM_WAVE(5, 2); break;
                case 6: FFMOE_GEMM_WAVE(6, 2); break;
                case 7: FFMOE_GEMM_WAVE(7, 2); break;
                case 8: FFMOE_GEMM_WAVE(8, 2); break;
                case 9: FFMOE_GEMM_WAVE(9, 3); break;
                case 10: FFMOE_GEMM_WAVE(10, 3); break;
                case 11: FFMOE_GEMM_WAVE(11, 3); break;
                case 12: FFMOE_GEMM_WAVE(12, 3); break;
                case 13: FFMOE_GEMM_WAVE(13, 4); break;
                case 14: FFMOE_GEMM_WAVE(14, 4); break;
                case 15: FFMOE_GEMM_WAVE(15, 4); break;
                default: FFMOE_GEMM_WAVE(16, 4); break;
            }
        }
#undef FFMOE_GEMM_WAVE
        if (!next.valid || gw.n_groups == 1) vmem_barrier<0>();     // (no load into LDS outlives the block)
        if (!next.valid) return;
        it = next;
    }
}

// ---------------------------------------------------------------------------------------------------
// Grouped product for chunks whose experts hold few pairs each (a short prompt): the GEMM's tiles and activation layout, N-blocks of
// four arena tiles, another way through them. There the expansion to 16-bit weights (68 vector instructions per 1 KiB tile of
// a wave, whatever the pairs, in front of its products) bounds the launch below about 50 pairs per expert: with the GEMMs that this
// form was built beside, 90 us for the 260 MB of a 37-row chunk's gate/up weights, 2.9 TB/s (here 47). Here a wave owns one arena tile row for the whole of K, streams its
// packed tiles through a ring of four and multiplies them in the offset form of the decode kernels (stream.hpp): about 52
// vector instructions per tile at 32 pairs, no expansion in LDS, the weights un-rounded. From two 16-pair blocks on the groups' input
// sums are made once per block of waves, each wave its share, and come in by outer products on the matrix unit: per 16 pairs, tile and
// group 80 cycles of it instead of 96, and 8 vector instructions instead of 16. The sums
// are the same and the order is a group's scale, then its bias (with the offset's correction): four groups' biases as one product of K = 4 would
// be 2 to 4 % faster again, but carries 128 times four groups' inputs in a sum at once, which is two bits less of it. 128 experts of
// 2,816 x 704, top-8, router table to combined rows, us with every wave's own sums | so: 301 rows 115.7 | 113.6, 448 rows 135.5 | 131.1,
// 576 rows 152.6 | 148.1, 736 rows 170.7 | 165.7 (FP16 123.7 | 121.9, 138.2 | 133.1, 159.4 | 156.8, 180.9 | 175.8); 64 of 320 x 192, 30
// pairs each, 17.8 | 18.4. The pairs' rows go straight into LDS, two groups at a time in a ring of four buffers (three for tiles of 64
// pairs, whose LDS is three blocks'), as lines of 128 bytes with their pieces turned by the row, so that every wave of the block
// reads the same fragments without conflicts and no register, store or address of theirs is on the waves' way; the weights stay in
// flight across the barriers, of which there is one per two groups. A step asks for its fragments in front of the 28 instructions that unpack its
// weights. (Rows through registers and two barriers, each fragment asked for where it is used: 248 vector instructions per four steps of
// 32 pairs, now 229. Three layers in turn, us of gate/up + down: 93 experts with 19 pairs each 55.5 + 31.1, now 50.9 + 30.5; 128 with 32
// 73.2 + 44.0 | 69.1 + 43.1, with 12 55.2 + 33.0 | 53.3 + 31.6, with 4 (tiles of 16) 48.5 + 29.7 | 48.9 + 28.4; a prompt of 301 rows 63.2 + 36.5 |
// 60.0 + 36.7. The same order of a step with the rows still through registers spills them: 48 experts with 19 pairs 33 -> 44 us.) What
// bounds it then is the weights' bytes (4.8 TB/s at 19 pairs with four blocks per unit) and the matrix and vector instructions
// together (64 pairs).
// A pair's arithmetic does not depend on its tile: any two launches of this kernel give the same row bit for bit.
// ---------------------------------------------------------------------------------------------------
constexpr int kStreamDepth = 4;                                             // weight tiles in flight per wave
constexpr int kStreamChunk = 2;                                             // groups per buffer of rows, and per barrier
constexpr uint32_t kStreamStageRow = 2 * kTilesPerBlock * kTileRows * 2 + 16;   // bytes: 128 output columns + padding

// The eight nibbles of a dword as matrix operands. bf16: 128 + q, as in the decode kernels. FP16: the subnormal q * 2^-24. With
// 1024 + q the fp32 sums of a group carry 1024 * sum x through their roundings, which made a 2,816-wide row's error against 64
// bits 3.60e-4 where the rounded weights of the GEMM have 3.58e-4.
template <bool F16>
__device__ __forceinline__ uint4 unpack8_stream(uint32_t w) {
    if constexpr (F16) return unpack8_fine<true>(w);
    else return unpack8_offset<false>(w);
}

// LDS of a block whose tiles have up to MAX_NM 16-pair blocks: buffers of a chunk of the pairs' rows each, then the groups' input sums.
template <int MAX_NM>
struct StreamLds {
    static constexpr int kBufs = MAX_NM <= 2 ? 4 : 3;                   // one in use, one whose sums are made, the others on their way
    static constexpr uint32_t kGroupBytes = 16 * MAX_NM * kGroup * 2, kBufBytes = kStreamChunk * kGroupBytes;
    static constexpr uint32_t kSumsAt = kBufs * kBufBytes, kBytes = kSumsAt + 2 * MAX_NM * kStreamChunk * 16 * 4;
};

template <bool GATE_UP, int NM, bool F16, bool ONCE, int MAX_NM>
__device__ __forceinline__ void stream_tile(const GemmWave &gw, const ArenaGeom &g, const TileSource &src, uint32_t tile0,
                                            uint8_t *lds, uint32_t lds_base, const uint32_t *__restrict__ sorted_token,
                                            const uint32_t *__restrict__ sorted_out_row, uint16_t *__restrict__ out,
                                            float *__restrict__ act_scale) {
    using L = StreamLds<MAX_NM>;
    constexpr int CHUNK = kStreamChunk, kAhead = L::kBufs - 1;
    static_assert(CHUNK == 2 && 2 * CHUNK % kStreamDepth == 0, "a group's ring slot follows from its place in a pair of chunks; two waves per group of a chunk");
    constexpr uint32_t kGroupBytes = NM * 2048;           // a group of the tile's rows in LDS
    const uint32_t lane = gw.lane, wave = gw.wave, j = lane & 15, jq = lane >> 4, tid = threadIdx.x;
    const uint32_t n_groups = gw.n_groups, last = n_groups - 1;
    const uint32_t n_chunks = (n_groups + CHUNK - 1) / CHUNK;
    static_assert(16 * NM * kStreamStageRow <= L::kSumsAt, "the down epilogue's rows fit in front of the sums");
    static_assert(NM * 2 * kWave * sizeof(uint4) + 4 * 16 * NM * sizeof(float) <= L::kSumsAt, "so do the activations and the peaks");

    // The pairs' rows go straight into LDS, 1 KiB per load, NM loads per wave and chunk. GATE_UP: eight rows of 128 bytes (one group),
    // eight neighbouring lanes per row; 16-byte piece c of row r lies at piece c ^ (r % 8), so that the sixteen rows of a fragment
    // fall on different banks. else: the activations are in fragment order already.
    const uint16_t *from[NM];
#pragma unroll
    for (int k = 0; k < NM; ++k) {
        const uint32_t piece = (wave + 4 * k) % (2 * NM);
        if constexpr (GATE_UP) {
            const uint32_t row = min(piece * 8 + (lane >> 3), gw.tile.rows - 1);
            from[k] = gw.a + (size_t)sorted_token[gw.tile.row_start + row] * gw.a_stride + 8 * ((lane & 7) ^ (lane >> 3));
        } else {
            from[k] = gw.a + ((size_t)(gw.act_block0 + (piece >> 1)) * n_groups * 2 + (piece & 1)) * (kWave * 8) + lane * 8;
        }
    }
    auto load_a = [&](uint32_t chunk, uint32_t buf) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < NM; ++k) {
            const uint32_t gl = (wave + 4 * k) / (2 * NM), piece = (wave + 4 * k) % (2 * NM);
            const uint32_t grp = min(chunk * CHUNK + gl, last);         // past the end: the last group again, never used
            global_to_lds_16(from[k] + (size_t)grp * (GATE_UP ? kGroup : 2 * kWave * 8), lds_base + buf + gl * kGroupBytes + piece * 1024);
        }
    };
    // fragment f of 16-pair block m, this lane's 16 bytes of it: k-half f % 2 (at0, at1) of group f / 2 of a chunk
    const uint32_t at0 = GATE_UP ? j * 128 + 16 * (jq ^ (j & 7)) : lane * 16, at1 = GATE_UP ? at0 ^ 64 : at0 + 1024;
    auto frag = [&](uint32_t at, int m, int gl) __attribute__((always_inline)) {
        return *reinterpret_cast<const uint4 *>(lds + at + gl * kGroupBytes + m * 2048);
    };

    uint4 ring_t[kStreamDepth];
    uint2 ring_s[kStreamDepth];
    auto fill = [&](int u, uint32_t grp) __attribute__((always_inline)) {
        const uint32_t tile = __builtin_amdgcn_readfirstlane(tile0 + min(grp, last));
        const u32x4_t t = __builtin_amdgcn_raw_buffer_load_b128(src.tiles, (int)(lane * 16u), (int)(tile * kTileBytes), ONCE ? kReadOnce : 0);
        const u32x2_t s = __builtin_amdgcn_raw_buffer_load_b64(src.scales, (int)(j * 8u), (int)(tile * kTileScaleBytes), 0);
        ring_t[u] = make_uint4(t.x, t.y, t.z, t.w);
        ring_s[u] = make_uint2(s.x, s.y);
    };
    constexpr int kFillLoads = 2;
    // the sums of two 16-pair blocks (or of the one): stream a and stream b of each, as the bias product's result has them
    constexpr bool kShared = NM > 1;
    constexpr int kPairs = (NM + 1) / 2;
    float __attribute__((ext_vector_type(kShared ? 16 : 8))) tot[kPairs];
#pragma unroll
    for (int i = 0; i < kPairs; ++i)
#pragma unroll
        for (int r = 0; r < (kShared ? 16 : 8); ++r) tot[i][r] = 0.0f;

    // The groups' input sums, a value per pair in LDS ([chunk % 2][16-pair block][group of the chunk][pair]): every wave makes its
    // share of a chunk's while the block is at the chunk before. (Of one 16-pair block every wave makes its own: two instructions
    // against a barrier, 37 rows of 128 experts 104.6 | 102.1 us.)
    float *const sums = reinterpret_cast<float *>(lds + L::kSumsAt);
    constexpr int kSums = (NM + 1) / 2;                   // 16-pair blocks per wave, of one of the chunk's two groups
    const uint32_t sum_gl = wave & 1;
    auto sum_block = [&](int k) __attribute__((always_inline)) { return min((wave >> 1) + 2u * k, NM - 1u); };
    uint4 sum_x[kSums][2];
    auto sum_read = [&](uint32_t buf) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < kSums; ++k) {
            const uint32_t here = buf + sum_gl * kGroupBytes + sum_block(k) * 2048;
            sum_x[k][0] = frag(at0 + here, 0, 0), sum_x[k][1] = frag(at1 + here, 0, 0);
        }
    };
    auto sum_up = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < kSums; ++k) {
            const f32x4 sx = group_input_sum<F16>(sum_x[k][0], sum_x[k][1]);
            if (j == 0) *reinterpret_cast<f32x4 *>(sums + ((slot * NM + sum_block(k)) * CHUNK + sum_gl) * 16 + 4 * jq) = sx;
        }
    };

    // One group. What it reads of LDS is asked for in front of the unpacking, which covers the way; the ring's slot is filled again behind it,
    // when its registers are free (`refills`: where it is wanted again). next_sums >= 0: on the way the wave's share of the next chunk's sums,
    // from buffer `next_buf`, for that slot.
    auto step = [&](uint32_t cur, uint32_t next_buf, int slot, int gl, int u, uint32_t refill, auto next_sums, auto refills) __attribute__((always_inline)) {
        constexpr int kNext = decltype(next_sums)::value;
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        uint4 x[2][2][2];                                   // of a pair of 16-pair blocks, and of the next pair
        auto read_x = [&](int i) __attribute__((always_inline)) {
#pragma unroll
            for (int q = 0; q < 2; ++q)
                if (2 * i + q < NM) x[i & 1][q][0] = frag(cur + at0, 2 * i + q, gl), x[i & 1][q][1] = frag(cur + at1, 2 * i + q, gl);
        };
        read_x(0);
        float both[kPairs];
#pragma unroll
        for (int i = 0; i < kPairs; ++i)
            if (kShared) both[i] = sums[((slot * NM + 2 * i) * CHUNK + gl) * 16 + (2 * i + 1 < NM ? (lane >> 5) * (CHUNK * 16) : 0) + j];
        if (kNext >= 0) sum_read(next_buf);
        __builtin_amdgcn_sched_barrier(0);
        const uint4 tile = ring_t[u];
        const uint2 sc = ring_s[u];
        const uint4 wa0 = unpack8_stream<F16>(tile.x), wa1 = unpack8_stream<F16>(tile.y);
        const uint4 wb0 = unpack8_stream<F16>(tile.z), wb1 = unpack8_stream<F16>(tile.w);
        float sa = bf16lo_to_f32(sc.x), sb = bf16lo_to_f32(sc.y), ta = bf16hi_to_f32(sc.x), tb = bf16hi_to_f32(sc.y);
        if constexpr (F16) {
            sa *= FineNibble<true>::kUnit;
            sb *= FineNibble<true>::kUnit;
        } else {
            ta = __builtin_fmaf(-Act<F16>::kOffset, sa, ta);
            tb = __builtin_fmaf(-Act<F16>::kOffset, sb, tb);
        }
        const float bias = jq & 1 ? tb : ta;
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (decltype(refills)::value) fill(u, refill);
#pragma unroll
        for (int i = 0; i < kPairs; ++i) {
            auto &t = tot[i];
            const int n = 2 * i + 1 < NM ? 2 : 1;
            if (i + 1 < kPairs) read_x(i + 1);
            f32x4 aa[2], ab[2], sx = zero;
            if (!kShared) sx = group_input_sum<F16>(x[0][0][0], x[0][0][1]);
#pragma unroll
            for (int q = 0; q < n; ++q) aa[q] = Act<F16>::mfma(x[i & 1][q][0], wa0, zero), ab[q] = Act<F16>::mfma(x[i & 1][q][0], wb0, zero);
#pragma unroll
            for (int q = 0; q < n; ++q) aa[q] = Act<F16>::mfma(x[i & 1][q][1], wa1, aa[q]), ab[q] = Act<F16>::mfma(x[i & 1][q][1], wb1, ab[q]);
            if (i == 0 && kNext >= 0) sum_up(kNext);
#pragma unroll
            for (int q = 0; q < n; ++q)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    t[8 * q + r] = __builtin_fmaf(sa, aa[q][r], t[8 * q + r]);
                    t[8 * q + 4 + r] = __builtin_fmaf(sb, ab[q][r], t[8 * q + 4 + r]);
                    if (!kShared) t[r] = __builtin_fmaf(ta, sx[r], t[r]), t[4 + r] = __builtin_fmaf(tb, sx[r], t[4 + r]);
                }
            // four outer products of 16 sums by 16 biases, lane (j, jq) has both for block jq: t + bias * sum, rounded once as by an fma
            if constexpr (kShared) t = __builtin_amdgcn_mfma_f32_16x16x1f32(both[i], bias, t, 0, 0, 0);
            // pinned: left alone, the compiler collects the scales' arithmetic of several groups and carries all
            // their matrix results there, which does not fit the register budget
            asm volatile("" : "+v"(t));
        }
    };

    // Chunk c lies in buffer c % kBufs. While the block is at it the loads of chunk c + kAhead go into the buffer of the chunk before, and
    // (kShared) chunk c + 1 is there already, for its sums. One barrier per chunk, at its end: it waits for the loads of the chunk
    // that is needed next, i.e. for all but those that every wave has asked for since: in the loop, and in front of it, always the same
    // number, chunk by chunk NM of rows, then one fill per group. The last one or two chunks, behind the loop, have nothing left to ask for (their rows
    // and weights went out kAhead chunks and kStreamDepth groups before), and their barriers wait for everything: a count over
    // refills that nobody reads would be wrong, since the compiler drops them.
    constexpr int kChunkFills = CHUNK * kFillLoads;
    constexpr int kInFlight = kShared ? kChunkFills * (kAhead - 1) + NM * (kAhead - 2) : kChunkFills * kAhead + NM * (kAhead - 1);
    static_assert(kStreamDepth == 2 * CHUNK, "two chunks' fills in front of the loop");
    uint32_t cur = 0, next_buf = L::kBufBytes;
#pragma unroll
    for (int a = 0; a < kAhead; ++a) {
        load_a(min((uint32_t)a, n_chunks - 1), a * L::kBufBytes);
        if (a >= kAhead - 2)
#pragma unroll
            for (int q = 0; q < CHUNK; ++q) fill((a - (kAhead - 2)) * CHUNK + q, (a - (kAhead - 2)) * CHUNK + q);
    }
    // (the first chunk, and kShared the second: less is in flight behind the first than there will be)
    ring_barrier<kShared ? (kAhead == 2 ? kChunkFills : 2 * kChunkFills + NM * (kAhead - 2)) : 2 * kChunkFills + NM * (kAhead - 1)>();
    if constexpr (kShared) {
        sum_read(0);
        sum_up(0);
        lds_barrier();
    }
    using Even = std::integral_constant<int, 0>;
    using Odd = std::integral_constant<int, 1>;
    using None = std::integral_constant<int, -1>;
    // a chunk; `asks`: of the loop. Behind it a chunk's second group may be missing.
    auto chunk = [&](uint32_t c, auto parity, auto asks) __attribute__((always_inline)) {
        constexpr int kParity = decltype(parity)::value;
        constexpr bool kAsks = decltype(asks)::value;
        using Sums = std::integral_constant<int, kShared ? kParity ^ 1 : -1>;
        if constexpr (kAsks) load_a(min(c + kAhead, n_chunks - 1), cur ? cur - L::kBufBytes : kAhead * L::kBufBytes);
        step(cur, next_buf, kParity, 0, (kParity * CHUNK) % kStreamDepth, c * CHUNK + kStreamDepth, Sums{}, asks);      // (past the last chunk sums nobody uses)
        if (kAsks || c * CHUNK + 1 < n_groups)
            step(cur, next_buf, kParity, 1, (kParity * CHUNK + 1) % kStreamDepth, c * CHUNK + 1 + kStreamDepth, None{}, asks);
        ring_barrier<kAsks ? kInFlight : 0>();
        cur = next_buf;
        next_buf = next_buf == kAhead * L::kBufBytes ? 0 : next_buf + L::kBufBytes;
    };
    uint32_t c = 0;
#pragma nounroll
    for (; (c + 2) * CHUNK <= n_groups; c += 2) {
        chunk(c, Even{}, std::true_type{});
        chunk(c + 1, Odd{}, std::true_type{});
    }
    if (c < n_chunks) chunk(c, Even{}, std::false_type{});
    if (c + 1 < n_chunks) chunk(c + 1, Odd{}, std::false_type{});
    ring_barrier<0>();                  // no load is on its way into what follows, and nobody reads the last chunk any more

    // lane (j, jq) holds, per stream, weight row j of the tile row for pairs 4 jq .. 4 jq + 3 of every 16-pair block
    uint16_t *half = reinterpret_cast<uint16_t *>(lds);
    if constexpr (GATE_UP) {
        float h[NM][4];
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) h[m][r] = gelu_tanh_fast(tot[m / 2][8 * (m & 1) + r]) * tot[m / 2][8 * (m & 1) + 4 + r];
        if constexpr (F16) {
            // the block scale of a pair's 64 activations, as in gemm_wave's epilogue: sixteen lanes hold a quarter of them
            float *peaks = reinterpret_cast<float *>(lds + NM * 2 * kFragBytes);        // [wave][pair]
#pragma unroll
            for (int m = 0; m < NM; ++m)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float v = fabsf(h[m][r]);
#pragma unroll
                    for (int x = 1; x < 16; x <<= 1) v = fmaxf(v, __shfl_xor(v, x, 64));
                    if (j == 0) peaks[wave * (16 * NM) + 16 * m + 4 * jq + r] = v;
                }
            lds_barrier();
#pragma unroll
            for (int m = 0; m < NM; ++m)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t pair = 16 * m + 4 * jq + r;
                    float peak = 0.0f;
#pragma unroll
                    for (int v = 0; v < 4; ++v) peak = fmaxf(peak, peaks[v * (16 * NM) + pair]);
                    int e = 0;
                    (void)frexpf(peak, &e);
                    e = max(e, -100);
                    h[m][r] *= ldexpf(1.0f, 14 - e);
                    if (wave == 0 && j == 0)
                        act_scale[((size_t)(gw.act_block0 + m) * g.gf + gw.nb) * 16 + 4 * jq + r] = ldexpf(1.0f, e - 14);
                }
        }
        // this wave's k = 16 wave + j of the block's group of F: k-half wave / 2, operand lane (pair, 2 (wave % 2) + j / 8)
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                half[((m * 2 + (wave >> 1)) * kWave + ((wave & 1) * 2 + (j >> 3)) * 16 + 4 * jq + r) * 8 + (j & 7)] = Act<F16>::round(h[m][r]);
        lds_barrier();
        for (uint32_t i = tid; i < (uint32_t)NM * 2 * kWave; i += 256) {
            const uint32_t m = i / (2 * kWave), at = i % (2 * kWave);
            *reinterpret_cast<uint4 *>(out + (((size_t)(gw.act_block0 + m) * g.gf + gw.nb) * 2 * kWave + at) * 8) = reinterpret_cast<const uint4 *>(lds)[i];
        }
        return;
    }
    uint8_t *rows = lds;
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t pair = 16 * m + 4 * jq + r;
            float va = tot[m / 2][8 * (m & 1) + r], vb = tot[m / 2][8 * (m & 1) + 4 + r];
            if constexpr (F16) {
                const float largest = act_scale[(size_t)gw.act_blocks * g.gf * 16 + (gw.act_block0 + m) * 16 + 4 * jq + r];
                va *= largest;
                vb *= largest;
            }
            uint16_t *dst = reinterpret_cast<uint16_t *>(rows + pair * kStreamStageRow) + 32 * wave + j;
            dst[0] = Act<F16>::round(va);
            dst[16] = Act<F16>::round(vb);
        }
    lds_barrier();
    const uint32_t piece = tid & 15;
    if (gw.nb * kTilesPerBlock + (piece >> 2) < gw.n_arena_tiles) {
#pragma unroll
        for (int k = 0; k < NM; ++k) {
            const uint32_t row = (tid >> 4) + 16 * k;
            if (row < gw.tile.rows)
                *reinterpret_cast<uint4 *>(out + (size_t)sorted_out_row[gw.tile.row_start + row] * g.d +
                                           gw.nb * (2 * kTilesPerBlock * kTileRows) + 8 * piece) =
                    *reinterpret_cast<const uint4 *>(rows + row * kStreamStageRow + 16 * piece);
        }
    }
}

// MAX_NM: 16-pair blocks of the largest tile the plan cut. `once_from`: with so many live experts or more the weights are read as data that no
// cache holds until the next call (read_once_experts), by tiles that are not whole: most are their expert's only one; the short one behind an
// expert's whole tiles reads so as well, which costs nothing in a layer that comes from memory (301 rows on 40 experts, three layers in turn, 83.5 us,
// 85.3 without; 700 Zipf rows of exponent 1.1 173.5 | 178). Not whole tiles, whose experts have others (the same Zipf rows with every tile so: 2 % slower).
template <bool GATE_UP, int MAX_NM, bool F16, int WAVES>
__global__ __launch_bounds__(256, WAVES) void prefill_stream_kernel(const PrefillPlan *__restrict__ plan, const PrefillTile *__restrict__ tiles,
                                                                    uint32_t n_nblocks, bool nb_major, uint32_t once_from, const uint8_t *__restrict__ arena_layer,
                                                                    const uint32_t *__restrict__ sorted_token,
                                                                    const uint16_t *__restrict__ a, uint32_t a_stride, uint32_t act_blocks,
                                                                    ArenaGeom g, const uint32_t *__restrict__ sorted_out_row,
                                                                    uint16_t *__restrict__ out, float *__restrict__ act_scale) {
    __shared__ __align__(16) uint8_t lds[StreamLds<MAX_NM>::kBytes];
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
    uint32_t ti, nb;
    if (!prefill_block(n_nblocks, nb_major, ti, nb) || ti >= plan->n_tiles) return;
    GemmWave gw;
    gw.tile = tiles[ti];
    gw.lane = threadIdx.x & 63;
    gw.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    gw.n_groups = GATE_UP ? g.gd : g.gf;
    gw.n_arena_tiles = GATE_UP ? g.gu_rb : g.dn_rbp;
    gw.nb = nb;
    gw.a = a;
    gw.a_stride = a_stride;
    gw.act_block0 = gw.tile.row_start / 16 + gw.tile.order;
    gw.act_blocks = act_blocks;
    // the tile row this wave multiplies; past the last one the last again (never stored)
    const uint32_t at = min(nb * kTilesPerBlock + gw.wave, gw.n_arena_tiles - 1);
    const uint8_t *expert_base = arena_layer + (size_t)__builtin_amdgcn_readfirstlane(gw.tile.expert) * g.expert_bytes;
    const size_t n_tiles = (size_t)gw.n_arena_tiles * gw.n_groups;
    const TileSource src = make_tile_source(expert_base + (GATE_UP ? g.gu_tiles_off : g.dn_tiles_off), n_tiles * kTileBytes,
                                            expert_base + (GATE_UP ? g.gu_scales_off : g.dn_scales_off), n_tiles * kTileScaleBytes);
    const uint32_t tile0 = at * gw.n_groups;
    const bool once = __builtin_amdgcn_readfirstlane(gw.tile.rows) < 16 * MAX_NM && plan->live_experts >= once_from;
#define FFMOE_STREAM(N)                                                                                                      \
    if constexpr (N <= MAX_NM) {                                                                                             \
        if (once) stream_tile<GATE_UP, N, F16, true, MAX_NM>(gw, g, src, tile0, lds, lds_base, sorted_token, sorted_out_row, out, act_scale);  \
        else stream_tile<GATE_UP, N, F16, false, MAX_NM>(gw, g, src, tile0, lds, lds_base, sorted_token, sorted_out_row, out, act_scale);      \
    }
    switch (__builtin_amdgcn_readfirstlane((gw.tile.rows + 15) / 16)) {
        case 1: FFMOE_STREAM(1); break;
        case 2: FFMOE_STREAM(2); break;
        case 3: FFMOE_STREAM(3); break;
        default: FFMOE_STREAM(4); break;
    }
#undef FFMOE_STREAM
}

// Between the two GEMMs of the FP16 prefill: a pair's blocks of 64 activations times their scales over its largest (powers of two),
// in place, and the largest behind the table at [n_pairs * blocks + pair] - what prefill_routed_down_tensorops does per
// threadgroup with `relative` and `pair_scale` as it takes the rows in (prefill.metal:731-741). Done there, every wave of the
// down products scaled every operand of its tile again: 8,000 pairs of 704 over 128 experts, down 82 us and this pass, scales
// only, 7 -> 68 + 10; the call with 62, 125 and 192 pairs per expert 215 -> 208, 301 -> 289 and 396 -> 375 us.
// PARTS waves per 16 pairs, each with every PARTS-th block of 64: the wave's first activations are on their way while the scales are
// read, whose largest meet in LDS. Where any of the 16 pairs is off its largest all of them are stored (times one: the same), as
// whole lines. Bound: memory's latency with few pairs, its rate with many. One wave per 16 pairs, skipping lanes | this: one expert,
// 512 rows, width 2,816 19.9 | 6.3 us, width 2,112 15.7 | 5.2, the calls 55.3 | 42.3 and 69.5 | 57.9; 3,072 rows top-8 of 128 of width 704 17.5 | 14.6.
// A layer of width 256 has nothing to share out and keeps one wave: 65,536 pairs, PARTS 4 | 2 | 1 14.3 | 12.6 | 11.8 us. There,
// with few columns in the down product (512), scaling in the products took 7 us less in all (of 135); at 2,816 columns it took more.
constexpr int kPairWaves = 4;                               // of a block
template <int PARTS>
__global__ __launch_bounds__(64 * kPairWaves) void prefill_pair_scale_kernel(const PrefillPlan *__restrict__ plan,
                                                                             const PrefillTile *__restrict__ tiles, uint32_t groups,
                                                                             uint32_t act_blocks, float *__restrict__ act_scale,
                                                                             uint16_t *__restrict__ acts) {
    __shared__ float peaks[kPairWaves][16];
    if (blockIdx.x >= plan->n_tiles) return;
    const PrefillTile tile = tiles[blockIdx.x];
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), part = wave % PARTS, j = lane & 15, jq = lane >> 4;
    const uint32_t in_tile = blockIdx.y * (kPairWaves / PARTS) + wave / PARTS;
    if (in_tile * 16 >= tile.rows) return;                  // (PARTS = 4: the whole block)
    const bool live = in_tile * 16 + j < tile.rows;
    const uint32_t block = tile.row_start / 16 + tile.order + in_tile;
    const float *const s = act_scale + (size_t)block * groups * 16 + j;
    uint4 *const a = reinterpret_cast<uint4 *>(acts) + (size_t)block * groups * (2 * kWave) + lane;
    constexpr int kAhead = PARTS == 1 ? 4 : 3;
    uint4 v[kAhead][2];
    float own[kAhead];
    auto load = [&](uint32_t b0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const uint32_t b = min(b0 + u * PARTS, groups - 1);            // past the last: read, not used
            v[u][0] = a[b * (2 * kWave)], v[u][1] = a[b * (2 * kWave) + kWave];
            own[u] = s[b * 16];
        }
    };
    load(part);
    float largest = 0.0f;
#pragma unroll 4
    for (uint32_t b = part * 4 + jq; b < groups; b += 4 * PARTS) largest = fmaxf(largest, s[b * 16]);
    largest = fmaxf(largest, __shfl_xor(largest, 16, 64));
    largest = fmaxf(largest, __shfl_xor(largest, 32, 64));
    if constexpr (PARTS > 1) {
        static_assert(PARTS == kPairWaves, "the waves of a block meet");
        if (jq == 0) peaks[wave][j] = largest;
        lds_barrier();
#pragma unroll
        for (int w = 0; w < PARTS; ++w) largest = fmaxf(largest, peaks[w][j]);
    }
    const float inv = 1.0f / largest;          // a scale is 2^(e - 14) with e >= -100: never zero
    for (uint32_t b0 = part; b0 < groups; b0 += kAhead * PARTS) {
        if (b0 != part) load(b0);
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const uint32_t b = b0 + u * PARTS;
            const float rel = live ? own[u] * inv : 1.0f;
            if (b >= groups || !__ballot(rel != 1.0f)) continue;
            const f16x2 r2 = __builtin_bit_cast(f16x2, Act<true>::pack(rel, rel));
            auto times = [&](uint32_t x) __attribute__((always_inline)) { return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, x) * r2); };
#pragma unroll
            for (int h = 0; h < 2; ++h)
                a[b * (2 * kWave) + h * kWave] = uint4{times(v[u][h].x), times(v[u][h].y), times(v[u][h].z), times(v[u][h].w)};
        }
    }
    if (live && jq == 0 && part == 0) act_scale[(size_t)act_blocks * groups * 16 + block * 16 + j] = largest;
}

// h2[t][c] = bf16(sum_r w[t][r] * partial[t][r][c]) over the routes the sort kept, fma in rank order
// (prefill.metal:544-565); dropped routes (zero weight, expert out of range) add nothing, which equals
// the reference's zero-filled partial rows without having to clear 138 MB first.
// TOP_K rows per token and no more, and of those the live ones: what a thread does not ask for is worth more than the round trip that asking
// for all eight places beside the weights and experts saves. us, 8,192 rows of 2,816, all live | half lost | seven eighths lost, so: top-8 64.5 | 37.6 |
// 15.3, top-2 21.3 | 14.5 | 10.6, top-1 15.0 | 11.3 | 9.8; all eight at once 61.5 | 61.5 | 65.5, 36.6 | 36.5 | 35.4, 30.2 | 31.2 | 31.4. 3,072 rows, top-8
// 23.1 | 14.0 | 7.3 (23.2 | 25.1 | 26); 301 rows 4.1 (4.3). The rows are read once, and said to be so: 8,192 rows, top-8, 91 without. Bound: the rows'
// bytes (6.4 TB/s at 8,192 rows, 6.7 from the caches at 3,072).
template <bool F16, int TOP_K>
__global__ __launch_bounds__(256) void prefill_combine_kernel(const uint16_t *__restrict__ partials,
                                                              const uint16_t *__restrict__ w, const uint32_t *__restrict__ idx,
                                                              uint32_t n_experts, uint32_t d, uint32_t t,
                                                              uint16_t *__restrict__ y) {
    // one thread per 16-byte piece of an output row, pieces numbered across rows so that every block is full
    const uint32_t pieces = d / 8, piece = blockIdx.x * 256 + threadIdx.x;
    const uint32_t tok = piece / pieces, c = (piece % pieces) * 8;
    if (tok >= t) return;
    uint16_t wbits[TOP_K];
    uint32_t expert[TOP_K];
#pragma unroll
    for (uint32_t r = 0; r < TOP_K; ++r) {
        wbits[r] = w[tok * TOP_K + r];
        expert[r] = idx[tok * TOP_K + r];
    }
    float wv[TOP_K];
    bool live[TOP_K];
#pragma unroll
    for (uint32_t r = 0; r < TOP_K; ++r) {
        live[r] = (wbits[r] & 0x7FFFu) != 0 && expert[r] < n_experts;
        wv[r] = Act<F16>::widen(wbits[r]);
    }
    uint4 p[TOP_K];
#pragma unroll
    for (uint32_t r = 0; r < TOP_K; ++r)
        if (live[r])
            p[r] = __builtin_bit_cast(uint4, __builtin_nontemporal_load(reinterpret_cast<const u32x4_t *>(partials + (size_t)(tok * TOP_K + r) * d + c)));
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (uint32_t r = 0; r < TOP_K; ++r) {
        if (live[r]) {
            const uint32_t pw[4] = {p[r].x, p[r].y, p[r].z, p[r].w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                acc[2 * i] = __builtin_fmaf(wv[r], Act<F16>::lo(pw[i]), acc[2 * i]);
                acc[2 * i + 1] = __builtin_fmaf(wv[r], Act<F16>::hi(pw[i]), acc[2 * i + 1]);
            }
        }
    }
    uint4 o;
    o.x = Act<F16>::pack(acc[0], acc[1]);
    o.y = Act<F16>::pack(acc[2], acc[3]);
    o.z = Act<F16>::pack(acc[4], acc[5]);
    o.w = Act<F16>::pack(acc[6], acc[7]);
    *reinterpret_cast<uint4 *>(y + (size_t)tok * d + c) = o;
}

// One pair of expert `expert` sent through the gate/up (or down) GEMM with the weight fragments copied out.
__global__ void prefill_dump_plan_kernel(uint32_t expert, PrefillPlan *plan, PrefillTile *tiles, uint32_t *sorted_token,
                                         uint32_t *sorted_out_row) {
    plan->n_pairs = 1;
    plan->n_tiles = 1;
    plan->live_experts = 1;
    PrefillTile tl;
    tl.expert = expert;
    tl.row_start = 0;
    tl.rows = 1;
    tl.order = 0;
    tiles[0] = tl;
    sorted_token[0] = 0;
    sorted_out_row[0] = 0;
}

// Pairs per M-tile of the grouped GEMMs: 256, or fewer where the gate/up items of the whole chunk then still run at once, a
// compute unit each - few experts leave most units idle otherwise. From the chunk's size alone: an expert's pairs are taken as
// normal about the mean with its root as deviation, so it has `full` whole tiles on average and one more with the rest. What
// an item takes is what dense_tile_rows has measured; where the down product's items take two rounds, the second begins on the
// units that had the smallest of the first. (Simulated for 19 shapes of 2 to 256 experts at 49 to 2,000 pairs per expert: 1 %
// off the best on average, worse than 256 pairs at two points.) Router table to combined rows, us at 256 pairs | the rule's, bf16
// (FP16): 8 experts of 4,096 x 1,536, 96 pairs each 86 | 68 (105 | 92), 192 pairs 108 | 89 (130 | 105); 8 of 2,048 x 704, 256 pairs
// 75 | 49 (88 | 61); 16 of 2,816 x 704, 192 pairs 82 | 75 (97 | 86). (Blocks of four waves, two to a unit, as the GEMMs had them
// before, took 80, 103, 68 and 84 there, in FP16 96, 122, 80 and 94.)
uint32_t gemm_tile_rows(uint32_t n_items, uint32_t n_experts, const ArenaGeom &g, uint32_t n_cus, uint32_t max_tiles) {
    const float mean = (float)n_items / n_experts, dev = sqrtf(mean), cus = (float)n_cus;
    const float nb_gu = (float)((g.gu_rb + kGemmTiles - 1) / kGemmTiles), nb_dn = (float)((g.dn_rbp + kGemmTiles - 1) / kGemmTiles);
    // Where a layer makes two rounds of items at most, no more than an expert of a uniform chunk would have: a skewed chunk's heavy
    // experts are then cut into items that run beside each other, a uniform chunk's tiles stay what they are. At 256 | so, us, Zipf
    // of exponent 1.1 (0.6): 64 experts of 1,024 x 512, 48 pairs each, FP16 67 | 60 (63 | 62); 256 of 512 x 256, 50 pairs 72 | 61
    // (73 | 62), 96 pairs 78 | 73 (78 | 74); 32 of 2,048 x 1,024, 62 pairs 82 | 74 (79 | 75); uniform routes within 1 %. Not where the
    // chip is full, where it expands the heavy experts' weights more often: 128 experts of 2,816 x 704, 62 pairs 211 | 248.
    const uint32_t most = n_experts * nb_gu <= 2 * cus ? (uint32_t)fminf((float)kBM, ceilf((mean + 4 * dev) / 16) * 16) : kBM;
    // Where the chip is full, 128, of which a compute unit works at two tiles at a time (GemmLds), as long as that holds nearly all of a
    // uniform chunk's experts whole; beyond, the second tiles' expansions cost more. us at 256 | 128, bf16 (FP16): 128 experts of
    // 2,816 x 704, 850 rows (53 pairs each) 182 | 164 (199 | 181), 1,000 179 | 167 (204 | 191), 1,500 (94) 214 | 203 (246 | 238), 1,792 (112)
    // 241 | 238 (275 | 272), 2,000 (125) 261 | 260 (289 | 299); Zipf of exponent 1.1, 1,000 rows 217 | 191 (236 | 216), 1,700 273 | 253 (305 |
    // 283), 3,072 (192) 377 | 386; 64 experts of 2,048 x 1,408, 94 pairs 152 | 140 (177 | 164), 112 171 | 165 (197 | 192), 141 188 | 210;
    // 256 of 512 x 256, 47 pairs 53 | 49 (62 | 58), Zipf 63 | 55 (73 | 64).
    if (n_items / (float)kBM * nb_gu > cus || n_experts * nb_gu > cus) {
        // (`most` and 256 fit every scratch, 128 where its tiles, one more than the whole ones per expert, do)
        const bool halves = mean + 1.5f * dev <= 128 && n_items / 128 + n_experts < max_tiles;
        return halves && most > 128 ? 128 : most;
    }
    uint32_t best = most;
    float least = 0.0f;
    for (uint32_t rows = most; rows >= 32; rows -= 16) {
        float full = floorf(fmaxf(mean - 4 * dev, 0.0f) / rows), variance = 0.0f;       // (every expert has these)
        for (float r = (full + 1) * rows; r < mean + 4 * dev; r += rows) {
            const float p = 0.5f * erfcf((r - mean) / (1.41421356f * dev));
            full += p, variance += p * (1 - p);
        }
        // (of a chunk's tiles, the number that three in five chunks stay below)
        const float tiles = n_experts * (full + 1) + 0.5f * sqrtf(n_experts * variance) - 0.3f;
        if (rows < most && (tiles * nb_gu > cus || n_items / rows + n_experts >= max_tiles)) continue;
        const float rest = fmaxf(mean - full * rows, 0.5f * dev), size_full = 10 + rows / 16.0f, size_rest = 10 + ceilf(rest / 16);
        const float largest = full > 0.02f ? size_full : 10 + ceilf(fminf((float)rows, mean + 2 * dev) / 16);
        auto rounds = [&](float nb) {
            const float n_full = n_experts * full * nb, n = n_full + n_experts * nb;
            if (tiles * nb <= cus) return largest;
            if (n > 2 * cus) return fmaxf(largest, (n_full * size_full + n_experts * nb * size_rest) / cus + 0.5f * size_full);
            if (n_full > cus) return 2 * size_full;
            return fmaxf(largest, n + n_full > 2 * cus ? size_full + size_rest : 2 * size_rest);
        };
        const float cost = rounds(nb_gu) * (g.gd + 6) + rounds(nb_dn) * (g.gf + 6);
        if (rows == most || cost < least * (best == most ? 0.99f : 1.0f)) least = cost, best = rows;
    }
    return best;
}

// Form and pairs per M-tile of a routed chunk. The line between prefill_stream_kernel and the GEMMs is drawn by the
// pairs per expert on average, from the chunk's size alone: the counts themselves are only known on the device, and a pair
// list's rows do not depend on how many of the chunk's pairs it names. Up to 28 the streaming product wins at every width.
// Beyond, up to 48: tiles of 32 pairs still where a tile from every expert would not fill the chip (its blocks then run at once,
// and a shorter tile is a shorter chain); tiles of 64 where K is long enough to pay for a block's start and end; else the
// grouped GEMMs, which have to expand little there. Router table to combined rows, us at 32 | 64 | 256 pairs per tile, bf16 (FP16):
// 128 experts, top-8, 2,816 x 704: 37 rows 97 | 101 | 143 (106 | 110 | 174), 301 rows 120 | 126 | 172 (130 | 137 | 191), 512 rows
// (32 pairs) 166 | 152 | 186 (178 | 165 | 203), 704 rows (44) 207 | 178 | 203 (220 | 192 | 215), 768 rows (48) 220 | 184 | 208
// (232 | 202 | 224), 1,000 rows (62, where many experts take two tiles) 218 | 220 | 219. 8 experts, 4,096 x 1,536: 28 pairs 56 | 62 | 69,
// 40 pairs 66 | 72 | 70 (76 | 87 | 83); 16 experts, 2,816 x 704, 48 pairs 54 | 55 | 54 (61 | 67 | 63). 64 experts, 1,024 x 512:
// 32 pairs 39 | 38 | 42 (49 | 45 | 48), 48 pairs 51 | 45 | 45 (57 | 53 | 51); 64 experts, 1,536 x 768, 48 pairs 77 | 71 | 74 (85 | 80 |
// 84); 256 experts, 512 x 256, 28 pairs 48 | 49 | 52, 40 pairs 59 | 56 | 53 (64 | 65 | 59).
// (The third figures are the four-wave GEMMs' that the line was drawn by; with a wave per arena tile they cross, at the first shape, at
// 44 pairs in FP16 - 42 pairs 182 | 184, 48 pairs 192 | 190 - and at some 40 in bf16, where the streamed weights are not rounded to 16
// bits: a chunk that had the smaller error keeps it.)
// Skewed routes move nothing: at the first shape with Zipf popularity of exponent 0.6, 1.1 and 1.6 the streaming form wins at
// every size up to 48 pairs (448 rows 146 | 159 | 166 against 186 | 201 | 196 for the GEMMs, 768 rows 192 | 201 | 212 against 225 |
// 226 | 232). Tiles of 128 lose everywhere (1,000 rows: 227, two waves per SIMD).
// Tiles of 16 pairs leave room for six blocks per compute unit (80 registers; FP16's epilogue does not fit them, and five blocks gain
// nothing): up to some five pairs per expert, where a tile from every expert is more blocks than four per unit and no more than six. Then
// a launch is one round instead of one and a part of one. us of the call at 32 | 16, bf16: 128 experts of 2,816 x 704, 17 rows 69.9 | 65.3,
// 24 rows 86 | 80.5, 37 rows 92.9 | 92.6, 64 rows 99.8 | 97.2, Zipf of exponent 1.1 48 rows 77.9 | 73.5, 80 rows 93.5 | 91.4, 128 rows (8
// pairs) 100.7 | 105.3; 64 of 2,048 x 1,408, 17 rows 58.7 | 56.4, 40 rows 67.6 | 66.9; 80 of 4,096 x 1,024, top-4, 80 rows 122 | 114. Past six
// blocks 256 of 2,816 x 704, 40 rows 125 | 127.5, 256 of 1,024 x 512, Zipf, 120 rows 44.0 | 46.0; below four 8 of 4,096 x 1,536, top-2, 18 rows
// 33.3 | 34.9, 64 of 2,048 x 704, Zipf, 64 rows 43.2 | 44.2.
struct TileForm {
    bool streamed;
    uint32_t rows;
};
TileForm prefill_tile_form(uint32_t n_items, uint32_t n_experts, const ArenaGeom &g, uint32_t n_nblocks, uint32_t n_cus, uint32_t max_tiles, bool f16) {
    // (1.32 tiles per expert at most, of the 2.5 that a scratch holds)
    if (!f16 && n_items <= 5 * n_experts && n_nblocks * n_experts > 4 * n_cus && n_nblocks * n_experts <= 6 * n_cus) return {true, 16};
    if (n_items <= 28 * n_experts) return {true, 32};
    if (n_items <= kPrefillStreamPairs * n_experts) {
        if (n_nblocks * n_experts <= n_cus) return {true, 32};
        if (n_items <= 32 * n_experts || g.d >= (f16 ? 1536u : 1024u)) return {true, 64};
    }
    return {false, gemm_tile_rows(n_items, n_experts, g, n_cus, max_tiles)};
}

// Rows per M-tile of a dense FFN's GEMMs: 16 n, n chosen so that the items fill their last round. A compute unit takes (10 + n) / 10 of
// about 1,000 cycles per group of an item and the time of some six groups around them; the lists' last N-blocks are counted as
// full ones. 2,816 -> 2,112 -> 2,816, us of the call at 256 rows per tile | the rule's: 102 | 62 at 897 rows (n = 4), 104 | 82 at
// 2,048 (9), 112 | 103 at 3,072 (13), 170 | 147 at 4,096 (12), 292 | 259 at 8,192 (13); FP16 inputs now 81, 105, 132,
// 179 and 311. Of n = 6..16 each, the rule's was the fastest at these sizes or within 3% of it. (All with one block per unit; up to 128 rows
// two of them run beside each other now: at 897 rows 52, FP16 66.)
uint32_t dense_tile_rows(uint32_t t, const ArenaGeom &g, uint32_t n_cus) {
    uint32_t best = kBM;
    uint64_t least = ~0ull;
    for (uint32_t n = kBM / 16; n >= 4; --n) {
        const uint32_t m = (t + 16 * n - 1) / (16 * n);
        auto rounds = [&](uint32_t arena_tiles) { return (uint64_t)((m * ((arena_tiles + kGemmTiles - 1) / kGemmTiles) + n_cus - 1) / n_cus); };
        const uint64_t cost = (10 + n) * (rounds(g.gu_rb) * (g.gd + 6) + rounds(g.dn_rbp) * (g.gf + 6));
        if (cost < least) least = cost, best = 16 * n;
    }
    return best;
}

// The same for a dense FFN's chunk that no bands took (at the model's widths FP16 beyond 384 rows, bf16 at 561 to 654 and beyond 704, where
// their rounds cost more; d or f beyond the bands' widths from 17 rows on): tiles of 32 rows while the gate/up
// launch is one round (four blocks per compute unit on the XCD with the most N-blocks), or while a chunk's products are few
// enough that it cost less than the GEMMs at 256 rows per tile did; at most kDenseTileStreamRows. With tiles of fewer rows the
// GEMMs are now the faster ones from some 640 rows on (2,816 -> 2,112, 897 rows 62 us, FP16 81, where 896 streamed ones take 78
// and 98), but their weights are rounded to 16 bits and the streamed ones' are not: a chunk that had the smaller error keeps it.
// us at 32 | 256 rows per tile, bf16 (FP16): 2,816 -> 2,112, 512 rows 54 | 78 (71 | 107), 800 rows 69 | 79 (88 | 108); 2,816 ->
// 2,816, 672 rows 70 | 87, 896 rows 94 | 88 (114 | 121); 4,096 -> 2,816, 672 rows 96 | 106, 896 rows 129 | 108 (147 | 142).
// Streamed tiles of 64 gain nothing (2,816 -> 2,112, 700 rows 71 | 66 at 32).
TileForm dense_tile_form(uint32_t t, const ArenaGeom &g, uint32_t n_nblocks, uint32_t n_cus, bool f16) {
    const bool one_round = (n_nblocks + 7) / 8 * ((t + 31) / 32) <= 4 * (n_cus / 8);
    if (t <= kDenseTileStreamRows && (one_round || (uint64_t)t * g.d * g.f <= (f16 ? 9600000000ull : 6600000000ull))) return {true, 32};
    return {false, dense_tile_rows(t, g, n_cus)};
}

// From how many live experts on a streamed chunk's weights are read once (kReadOnce): where those of all the context's layers, which a program
// takes one after the other, are more than the memory side's cache holds - this layer's live experts, which the device alone knows, taken for every
// layer's. Asked where the chunk's routes could reach more than the cache in this one layer. 128 experts of 2,816 x 704 (3.3 MB each), us of the call
// without | with the hint. Three layers in turn: 24 rows, 40 live 46.8 | 42.5; 37 rows, 40 live 44.4 | 39.7, 80 live 66.9 | 57.8; 100 rows, 60 live 58.1 |
// 53.1; 301 rows, 40 live 82.4 | 79.7, 110 live 103.0 | 96.6. One layer again and again, tiles of 32: 100 rows, 60 live 46.6 | 52.0, 80 live 58.1 | 61.0, 110 live
// 91 | 82; 301 rows, 60 live 79.8 | 84.8, 80 live 83.2 | 89.9, 110 live 102 | 97.6. Tiles of 16, six blocks per unit, lose their lines from three
// quarters of the cache on: 24 rows, 40 live 37.7 | 40.6, 58 live 48.3 | 48.5, 74 live 61.3 | 56.8; 37 rows, 50 live 45.3 | 46.5, 60 live 48.9 | 47.6, 79 live 61.4 | 57.6.
uint32_t read_once_experts(uint32_t n_items, uint32_t n_experts, uint32_t n_layers, const ArenaGeom &g, uint32_t tile_rows) {
    if ((size_t)min(n_items, n_experts) * g.expert_bytes <= kMemoryCacheBytes) return 0xFFFFFFFFu;
    const size_t holds = tile_rows == 16 ? kMemoryCacheBytes / 4 * 3 : kMemoryCacheBytes;
    return (uint32_t)(holds / ((size_t)n_layers * g.expert_bytes)) + 1;
}

template <bool GATE_UP>
auto stream_kernel(uint32_t tile_rows, bool f16) {
    if (tile_rows == 16) return prefill_stream_kernel<GATE_UP, 1, false, 6>;           // (bf16 alone: prefill_tile_form)
    if (tile_rows == 32) return f16 ? prefill_stream_kernel<GATE_UP, 2, true, 4> : prefill_stream_kernel<GATE_UP, 2, false, 4>;
    return f16 ? prefill_stream_kernel<GATE_UP, 4, true, 3> : prefill_stream_kernel<GATE_UP, 4, false, 3>;
}

}  // namespace

uint32_t prefill_dump_fragments(const ArenaGeom &g, bool gate_up) {
    const uint32_t tiles = gate_up ? g.gu_rb : g.dn_rbp, groups = gate_up ? g.gd : g.gf;
    return (tiles + kTilesPerBlock - 1) / kTilesPerBlock * groups * 16;
}

hipError_t launch_prefill_dump_tiles(hipStream_t s, const uint8_t *arena_layer, ArenaGeom g, uint32_t expert, bool gate_up,
                                     PrefillScratch sc, void *dump, bool f16, bool large_scales) {
    if (f16 && !sc.act_scale) return hipErrorInvalidValue;
    hipLaunchKernelGGL(prefill_dump_plan_kernel, dim3(1), dim3(1), 0, s, expert, sc.plan, sc.tiles, sc.sorted_token,
                       sc.sorted_out_row);
    if (large_scales)
        return launch_prefill_large_scale(s, arena_layer, g, gate_up, 1, gate_up ? sc.partials : sc.acts, g.d, gate_up ? sc.acts : sc.partials, sc, f16,
                                          dump);
    // the pair's input row is whatever row 0 of the scratch holds: only the weight side is looked at
#define FFMOE_DUMP(GU, H, A, STRIDE, OUT, NB)                                                                              \
    hipLaunchKernelGGL((prefill_gemm_kernel<GU, H, false, 4, true>), dim3((NB) * 8), dim3(64 * kGemmTiles), 0, s, arena_layer, g, sc.plan, sc.tiles,  \
                       sc.sorted_token, sc.sorted_out_row, A, STRIDE, OUT, false, sc.act_scale, sc.act_blocks, static_cast<uint4 *>(dump))
    if (gate_up) {
        const uint32_t nb = (g.gu_rb + kGemmTiles - 1) / kGemmTiles;
        if (f16) FFMOE_DUMP(true, true, sc.partials, g.d, sc.acts, nb); else FFMOE_DUMP(true, false, sc.partials, g.d, sc.acts, nb);
    } else {
        const uint32_t nb = (g.dn_rbp + kGemmTiles - 1) / kGemmTiles;
        if (f16) FFMOE_DUMP(false, true, sc.acts, g.f, sc.partials, nb); else FFMOE_DUMP(false, false, sc.acts, g.f, sc.partials, nb);
    }
#undef FFMOE_DUMP
    return hipGetLastError();
}

hipError_t launch_prefill(hipStream_t s, const uint8_t *arena_layer, ArenaGeom g, uint32_t n_experts, uint32_t top_k,
                          const uint16_t *x, uint32_t x_stride, uint32_t t, const uint32_t *idx, const uint16_t *w,
                          const ffmoe_pair *pairs, uint32_t n_pairs_in, uint16_t *y, uint16_t *partials_out,
                          PrefillScratch sc, KernelTimer *timer, uint32_t n_cus, uint32_t n_layers, bool f16, bool dense, bool large_scales) {
    // dense: the caller vouches for a dense FFN's chunk - one expert, top_k = 1, every row routed to it at weight 1
    dense = dense && n_experts == 1 && top_k == 1 && !pairs && !y;
    timer->begin(s);
    ItemSource src{};
    src.idx = pairs ? nullptr : idx;
    src.w = pairs ? nullptr : w;
    src.pairs = pairs;
    src.n_items = pairs ? n_pairs_in : t * top_k;
    src.top_k = top_k;
    src.n_experts = n_experts;
    src.t = t;
    if (src.n_items == 0) return hipSuccess;
    const uint32_t n_blocks = (src.n_items + kSortBlock - 1) / kSortBlock;
    const uint32_t nb_gu = (g.gu_rb + kTilesPerBlock - 1) / kTilesPerBlock, nb_dn = (g.dn_rbp + kTilesPerBlock - 1) / kTilesPerBlock;
    const TileForm form = dense ? dense_tile_form(t, g, nb_gu, n_cus, f16)
                                : prefill_tile_form(max(src.n_items, t * top_k), n_experts, g, nb_gu, n_cus, sc.max_tiles, f16);
    const bool streamed = form.streamed;
    const uint32_t tile_rows = form.rows;
    if (dense) {
        hipLaunchKernelGGL(prefill_dense_plan_kernel, dim3(n_blocks), dim3(kSortBlock), 0, s, t, tile_rows, sc.plan, sc.tiles, sc.sorted_token,
                           sc.sorted_out_row);
    } else {
        if (src.n_items <= sort_one_launch(src)) {
            hipLaunchKernelGGL(prefill_sort_kernel, dim3(n_experts), dim3(sort_threads(src.n_items)), 0, s, src, sc.plan, sc.tiles, sc.max_tiles,
                               TileRows(tile_rows), sc.sorted_token, sc.sorted_out_row);
        } else {
            hipLaunchKernelGGL(prefill_hist_kernel, dim3(n_blocks), dim3(kSortBlock), 0, s, src, sc.block_cnt);
            uint32_t e_pad = 1;
            while (e_pad < n_experts) e_pad <<= 1;      // n_experts <= FFMOE_MAX_EXPERTS = 256 <= kScanThreads
            const uint32_t run = (n_blocks + kScanThreads / e_pad - 1) / (kScanThreads / e_pad);     // sort blocks per thread
            hipLaunchKernelGGL((run <= 16 ? prefill_scan_kernel<16> : prefill_scan_kernel<32>), dim3(1), dim3(kScanThreads), 0, s, n_blocks,
                               n_experts, e_pad, sc.block_cnt, sc.plan, sc.tiles, sc.max_tiles, TileRows(tile_rows));
            hipLaunchKernelGGL(prefill_scatter_kernel, dim3(n_blocks), dim3(kSortBlock), 0, s, src, sc.block_cnt, sc.sorted_token,
                               sc.sorted_out_row);
        }
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    timer->mark(s, FFMOE_K_PREFILL_SORT);
    const uint32_t tile_cap = min(sc.max_tiles, dense ? (t + tile_rows - 1) / tile_rows : src.n_items / tile_rows + n_experts);
    const uint32_t tile_slots = (tile_cap + 7) / 8 * 8;
    if (f16 && !sc.act_scale) return hipErrorInvalidValue;      // allocated when the context was switched to FP16
    // grid: (N-blocks x tile slots) in either order of the kernel's block map
    const bool nb_major = n_experts == 1;
    auto grid_of = [&](uint32_t n_nblocks) { return nb_major ? 8 * ((n_nblocks + 7) / 8) * tile_cap : n_nblocks * tile_slots; };
    const uint32_t gemm_gu = (g.gu_rb + kGemmTiles - 1) / kGemmTiles, gemm_dn = (g.dn_rbp + kGemmTiles - 1) / kGemmTiles;
    uint16_t *partials = partials_out ? partials_out : sc.partials;
    float *act_scale = f16 ? sc.act_scale : nullptr;
    const uint32_t act_blocks = f16 ? sc.act_blocks : 0u;
    // (a row's address is 32 bits from the first row's where that reaches the last)
    const bool wide = (uint64_t)t * x_stride * 2 > 0xFFFFFFFFull;
    const uint32_t once_from = read_once_experts(src.n_items, n_experts, n_layers, g, tile_rows);
    // Tiles of up to 128 pairs run two blocks to a compute unit (GemmLds), also where a launch has no more items than units and every block
    // is alone: the shorter start and end of an item are worth 1 to 8 % there. Not tiles of 112 pairs (FP16: 96 and 112) over 40 groups and
    // more: alone, the longer rings and queues win. us of the call with two blocks | one, dense: 4,096 -> 1,408, FP16, 1,536 rows (96 each)
    // 84.7 | 79.5, 2,048 rows (128) 91 | 95; 2,816 -> 2,816, FP16, 897 rows (96) 84.1 | 81.6, 1,200 rows (112) 92.5 | 89.5, bf16 77.4 | 75.9; 2,816 -> 704,
    // FP16, 2,048 rows (96) 60.5 | 56.5; 2,048 -> 1,408, 1,536 rows (80) 44.3 | 45.2; 1,024 -> 512, 897 rows (64) 23.5 | 24.5, FP16 30.2 | 31.3. 8 experts
    // of 4,096 x 1,536, 192 pairs each (112) 89.1 | 87.6, FP16 107.5 | 103.9, 96 pairs each (64), FP16, 78.5 | 80.1.
    const auto two_blocks = [&](uint32_t groups, uint32_t n_nb) {
        return tile_rows <= 128 && (groups < 40 || tile_cap * n_nb > n_cus || tile_rows <= (f16 ? 80u : 96u) || tile_rows == 128);
    };
#define FFMOE_GEMM_LC(GU, A, STRIDE, OUT, NB, LC)                                                                             \
    hipLaunchKernelGGL((GU && wide ? (f16 ? prefill_gemm_kernel<GU, true, GU, LC> : prefill_gemm_kernel<GU, false, GU, LC>)   \
                                   : (f16 ? prefill_gemm_kernel<GU, true, false, LC> : prefill_gemm_kernel<GU, false, false, LC>)), \
                       dim3(8 * min((GemmLds<LC>::kBlocks * n_cus + 7) / 8, tile_slots * (NB))), dim3(64 * kGemmTiles), 0, s, \
                       arena_layer, g, sc.plan, sc.tiles, sc.sorted_token, sc.sorted_out_row, A, STRIDE, OUT, nb_major,    \
                       act_scale, act_blocks, nullptr)
#define FFMOE_GEMM(GU, A, STRIDE, OUT, NB)                                                                                    \
    do {                                                                                                                      \
        if (two_blocks(GU ? g.gd : g.gf, NB)) FFMOE_GEMM_LC(GU, A, STRIDE, OUT, NB, 2);                                       \
        else FFMOE_GEMM_LC(GU, A, STRIDE, OUT, NB, 4);                                                                        \
    } while (0)
#define FFMOE_STREAM(GU, A, STRIDE, OUT, NB)                                                                                  \
    hipLaunchKernelGGL(stream_kernel<GU>(tile_rows, f16), dim3(grid_of(NB)), dim3(256), 0, s, sc.plan, sc.tiles, NB,    \
                       nb_major, once_from, arena_layer, sc.sorted_token, A, STRIDE, act_blocks, g, sc.sorted_out_row, OUT, act_scale)
    if (large_scales) {
        if ((e = launch_prefill_large_scale(s, arena_layer, g, true, tile_cap, x, x_stride, sc.acts, sc, f16)) != hipSuccess) return e;
    } else if (streamed) FFMOE_STREAM(true, x, x_stride, sc.acts, nb_gu);
    else FFMOE_GEMM(true, x, x_stride, sc.acts, gemm_gu);
    timer->mark(s, FFMOE_K_PREFILL_GATE_UP);
    if (f16) {
        const bool one = g.gf <= 4;
        hipLaunchKernelGGL((one ? prefill_pair_scale_kernel<1> : prefill_pair_scale_kernel<kPairWaves>),
                           dim3(tile_cap, one ? (tile_rows / 16 + kPairWaves - 1) / kPairWaves : tile_rows / 16), dim3(64 * kPairWaves), 0, s,
                           sc.plan, sc.tiles, g.gf, sc.act_blocks, sc.act_scale, sc.acts);
    }
    if (large_scales) {
        if ((e = launch_prefill_large_scale(s, arena_layer, g, false, tile_cap, sc.acts, g.f, partials, sc, f16)) != hipSuccess) return e;
    } else if (streamed) FFMOE_STREAM(false, sc.acts, g.f, partials, nb_dn);
    else FFMOE_GEMM(false, sc.acts, g.f, partials, gemm_dn);
#undef FFMOE_GEMM
#undef FFMOE_STREAM
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    timer->mark(s, FFMOE_K_PREFILL_DOWN);
    if (y) {
        auto launch = [&](auto k) {
            constexpr int K = decltype(k)::value;
            hipLaunchKernelGGL((f16 ? prefill_combine_kernel<true, K> : prefill_combine_kernel<false, K>), dim3((t * (g.d / 8) + 255) / 256), dim3(256), 0, s,
                               partials, w, idx, n_experts, g.d, t, y);
        };
        using std::integral_constant;
        switch (top_k) {
            case 1: launch(integral_constant<int, 1>{}); break;
            case 2: launch(integral_constant<int, 2>{}); break;
            case 3: launch(integral_constant<int, 3>{}); break;
            case 4: launch(integral_constant<int, 4>{}); break;
            case 5: launch(integral_constant<int, 5>{}); break;
            case 6: launch(integral_constant<int, 6>{}); break;
            case 7: launch(integral_constant<int, 7>{}); break;
            default: launch(integral_constant<int, 8>{}); break;        // (top_k <= 8: checked where a context is made)
        }
        timer->mark(s, FFMOE_K_PREFILL_COMBINE);
    }
    timer->finish();
    return hipGetLastError();
}

}  // namespace ffmoe
