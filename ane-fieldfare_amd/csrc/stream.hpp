// Register-ring streaming of two-stream arena tiles, shared by the expert kernels and the resident-matrix
// GEMV: one wave consumes a group's tile (16 + 16 weight rows x 64 k) against up to 16 token rows on the
// matrix unit and immediately starts the load that refills the ring slot.
#pragma once

#include "common.hpp"

namespace ffmoe {

constexpr int kKSplit = 4;      // waves of a block that split K
constexpr int kRing = 11;       // groups in flight per wave (= one K-slice of D = 2816)

struct TwoStreamAcc {
    f32x4 a, b;
};

struct WeightRing {
    uint4 t[kRing];
    uint2 s[kRing];
};

// Where a wave's tiles come from: two buffer descriptors (scalar registers). A ring load is then a single
// buffer_load with the lane's fixed 32-bit offset and a scalar byte offset - no per-load 64-bit address
// arithmetic in vector registers, which otherwise costs two registers per load in flight - and a load
// past the end of the region returns zero instead of faulting.
struct TileSource {
    __amdgpu_buffer_rsrc_t tiles, scales;
};

__device__ __forceinline__ TileSource make_tile_source(const uint8_t *tiles, size_t tile_bytes, const uint8_t *scales,
                                                       size_t scale_bytes) {
    TileSource src;
    src.tiles = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(tiles), 0, (int)(uint32_t)tile_bytes, 0x00020000);
    src.scales = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(scales), 0, (int)(uint32_t)scale_bytes, 0x00020000);
    return src;
}

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

// For tiles that no other block counts on and no cache holds until the next call: the load's non-temporal bit. The memory side's cache has
// 256 MB; a sweep of more pushes its own lines out before they are wanted again, and is the faster when it leaves none there: the
// head's 415 MB, one input row, with the draw behind it 89.0 -> 79.8 us, greedy 84.7 -> 78.4; the layer of a 37-row prompt (a chunk's 390 MB of experts)
// 126.1 -> 116.2, of 301 rows 177 -> 169.6. Below that the next call finds the lines: a matrix of 158 MB 26.5 us, so 28.1; of 25 MB 6.9 | 8.7 (a
// layer's experts: read_once_experts in prefill.hip).
constexpr int kReadOnce = 2;
constexpr size_t kMemoryCacheBytes = 256u << 20;

// `tile_index` = index of the 1 KiB tile inside the region (wave-uniform). ONCE: see kReadOnce.
template <bool ONCE = false>
__device__ __forceinline__ void ring_fill(WeightRing &ring, int u, const TileSource &src, uint32_t tile_index,
                                          uint32_t lane) {
    // the index is wave-uniform by contract; pinning it to a scalar register spares the waterfall loop the
    // compiler emits whenever it happened to compute a uniform value in a vector register
    tile_index = __builtin_amdgcn_readfirstlane(tile_index);
    const u32x4_t t = __builtin_amdgcn_raw_buffer_load_b128(src.tiles, (int)(lane * 16u), (int)(tile_index * kTileBytes), ONCE ? kReadOnce : 0);
    const u32x2_t s = __builtin_amdgcn_raw_buffer_load_b64(src.scales, (int)((lane & 15u) * 8u),
                                                           (int)(tile_index * kTileScaleBytes), 0);
    ring.t[u] = make_uint4(t.x, t.y, t.z, t.w);
    ring.s[u] = make_uint2(s.x, s.y);
}

// The same where it stands, before what follows: for the fills in front of a loop of ring_steps, whose waits count on the loads' order.
template <bool ONCE = false>
__device__ __forceinline__ void ring_fill_here(WeightRing &ring, int u, const TileSource &src, uint32_t tile_index, uint32_t lane) {
    ring_fill<ONCE>(ring, u, src, tile_index, lane);
    __builtin_amdgcn_sched_barrier(0);
}

// The lane of a refill that is not wanted: its tile's bytes lie 2 GiB further on, past the end of a region of less (kNoLaneTiles), and memory is
// not asked for them. (Its scales, 128 bytes, are read and left.) The offset is the lane's own, which is held against what the descriptor has
// left behind the tile's; with the tile's it stays below 4 GiB.
constexpr uint32_t kNoLaneTiles = (1u << 31) / kTileBytes;
__device__ __forceinline__ uint32_t no_lane(uint32_t lane) { return lane | 0x08000000u; }

// Sum of a group's 64 inputs per token column, in the register layout of the matrix results: the product
// with an all-ones operand. It depends on the token operand only, so a wave that walks several tile rows
// with the same operand computes it once per group, not once per tile.
template <bool F16 = false>
__device__ __forceinline__ f32x4 group_input_sum(const uint4 &x0, const uint4 &x1) {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    const uint4 ones = {Act<F16>::kOnesBits, Act<F16>::kOnesBits, Act<F16>::kOnesBits, Act<F16>::kOnesBits};
    return Act<F16>::mfma(x1, ones, Act<F16>::mfma(x0, ones, zero));
}

// Consume ring slot u against the resident token operand (`sx` = its group_input_sum), then start the load
// that refills the slot (REFILL = false: a wave that walks one tile row only has nothing to refill).
// SUMS: of the lane's four results, how many are kept up.
// PIN: the refill stands behind the unpacking of its slot, and nowhere else. Left alone the compiler collects the refills of a whole tile row at its
// end and waits for nearly all of them at the next one's start, so that a wave has its twelve KiB in flight a part of the time only. Us of a call as the compiler
// has it | pinned, both builds in turn, weights of two heads or three layers in turn: 262,144 x 2,816, greedy with confidence, 16 rows 73.3 | 71.3; fp32 logits of
// 1 row 64.2 | 60.8, of 16 rows 75.1 | 71.0; verify block of 16 rows 46.4 | 45.2, layer block of 1 row 28.9 | 28.3, of 5 FP16 rows 43.5 | 43.3 (three runs of a side
// differ by 0.1, the heads' by 0.5); a dense FFN with skinny_down_ksplit_persistent alone changed, 48 layers in turn, 2,816 -> 2,112, 1 row 11.76 | 11.57,
// 16 rows 12.67 | 12.55, 2,816 -> 2,816, 1 row 12.12 | 11.86. Not for a wave of one tile row, whose rows and weights are better asked for as the compiler has it
// (skinny_down_lds: 5.9 us at 1 row, pinned 6.2 to 6.5) or which refills nothing (decode_down_combine_kernel: REFILL = false). The last tile row's refills come with
// no_lane (asked for once more, its tiles are the launch's last requests: layer block of 1 row 28.7 | 28.3, a sampled head's row 74.9 | 73.0); written as steps
// without a refill, behind a branch, the compiler keeps both rows' operands and spills.
template <bool F16 = false, bool REFILL = true, int SUMS = 4, bool ONCE = false, bool PIN = REFILL>
__device__ __forceinline__ void ring_step(WeightRing &ring, int u, bool live, const uint4 &x0, const uint4 &x1,
                                          const f32x4 &sx, TwoStreamAcc &tot, const TileSource &src,
                                          uint32_t next_tile_index, uint32_t lane) {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    const uint4 tile = ring.t[u];
    uint2 sc = ring.s[u];
    if (!live) sc = make_uint2(0u, 0u);
    if (REFILL && !PIN) ring_fill<ONCE>(ring, u, src, next_tile_index, lane);
    const uint4 wa0 = unpack8_offset<F16>(tile.x), wa1 = unpack8_offset<F16>(tile.y), wb0 = unpack8_offset<F16>(tile.z), wb1 = unpack8_offset<F16>(tile.w);
    if (PIN) {
        __builtin_amdgcn_sched_barrier(0);
        ring_fill_here<ONCE>(ring, u, src, next_tile_index, lane);
    }
    f32x4 acc_a = Act<F16>::mfma(x0, wa0, zero);
    acc_a = Act<F16>::mfma(x1, wa1, acc_a);
    f32x4 acc_b = Act<F16>::mfma(x0, wb0, zero);
    acc_b = Act<F16>::mfma(x1, wb1, acc_b);
    const float sa = bf16lo_to_f32(sc.x), ba = bf16hi_to_f32(sc.x);
    const float sb = bf16lo_to_f32(sc.y), bb = bf16hi_to_f32(sc.y);
    const float ta = __builtin_fmaf(-Act<F16>::kOffset, sa, ba), tb = __builtin_fmaf(-Act<F16>::kOffset, sb, bb);
#pragma unroll
    for (int r = 0; r < SUMS; ++r) {
        tot.a[r] = __builtin_fmaf(sa, acc_a[r], tot.a[r]);
        tot.a[r] = __builtin_fmaf(ta, sx[r], tot.a[r]);
        tot.b[r] = __builtin_fmaf(sb, acc_b[r], tot.b[r]);
        tot.b[r] = __builtin_fmaf(tb, sx[r], tot.b[r]);
    }
}

// A wave's share of K when the four waves of a block split it.
struct KSlice {
    uint32_t g0, ng, g_last;      // first group, number of groups, last valid group of this wave's share of K
};
__device__ __forceinline__ KSlice k_slice(uint32_t groups, uint32_t ks) {
    const uint32_t per = (groups + kKSplit - 1) / kKSplit;
    const uint32_t g0 = min(ks * per, groups), g1 = min(groups, g0 + per);
    return KSlice{g0, g1 - g0, g1 > g0 ? g1 - 1 : groups - 1};
}

// The token operand is the call's rows themselves, row min(j, rows - 1) in token column j (in the expert kernels:
// which expert a block serves does not matter for fetching them, so they can be requested before the routes are
// known; an expert's routes only decide which columns of the result are stored).
// Load layout: four neighbouring lanes read 64 contiguous bytes of one row (row lane / 4, 8-element chunk
// lane % 4), 16 requests of 64 bytes per instruction; with the matrix unit's own layout (row lane % 16)
// every lane would be a request of its own and the 22 loads of a wave would keep the address unit busy
// for microseconds. turn_token_rows() re-lays them into the operand layout (lane (j, jq): row j, chunk jq).
__device__ __forceinline__ void load_token_rows(const uint16_t *__restrict__ x, uint32_t x_stride, uint32_t rows,
                                                uint32_t lane, const KSlice &k, uint4 (&x0)[kRing], uint4 (&x1)[kRing]) {
    const uint16_t *xrow = x + (size_t)min(lane >> 2, rows - 1) * x_stride + 8 * (lane & 3);
#pragma unroll
    for (int u = 0; u < kRing; ++u) {
        const bool live = (uint32_t)u < k.ng;
        const uint32_t gg = min(k.g0 + u, k.g_last);
        x0[u] = live ? *reinterpret_cast<const uint4 *>(xrow + gg * kGroup) : uint4{0, 0, 0, 0};
        x1[u] = live ? *reinterpret_cast<const uint4 *>(xrow + gg * kGroup + 32) : uint4{0, 0, 0, 0};
    }
}

// Up to four rows straight in the operand layout, row t as operand row 4 t (and 4 t + 1 .. + 3, whose results nobody keeps): the
// lanes of a row and quarter ask for the same 16 bytes, so an instruction is as many requests of 64 bytes as there are rows.
__device__ __forceinline__ void load_few_rows(const uint16_t *__restrict__ x, uint32_t x_stride, uint32_t rows, uint32_t lane,
                                              const KSlice &k, uint4 (&x0)[kRing], uint4 (&x1)[kRing]) {
    const uint16_t *xrow = x + (size_t)min((lane & 15) >> 2, rows - 1) * x_stride + 8 * (lane >> 4);
#pragma unroll
    for (int u = 0; u < kRing; ++u) {
        const bool live = (uint32_t)u < k.ng;
        const uint32_t gg = min(k.g0 + u, k.g_last);
        x0[u] = live ? *reinterpret_cast<const uint4 *>(xrow + gg * kGroup) : uint4{0, 0, 0, 0};
        x1[u] = live ? *reinterpret_cast<const uint4 *>(xrow + gg * kGroup + 32) : uint4{0, 0, 0, 0};
    }
}

template <int N> __device__ __forceinline__ void turn_token_rows(uint32_t lane, uint4 (&x0)[N], uint4 (&x1)[N]) {
    const uint32_t j = lane & 15, jq = lane >> 4;
    const int pull = (int)((4 * j + jq) * 4);       // operand lane (j, jq) takes what load lane 4 j + jq holds
    auto turn = [&](uint4 &v) {
        v.x = (uint32_t)__builtin_amdgcn_ds_bpermute(pull, (int)v.x);
        v.y = (uint32_t)__builtin_amdgcn_ds_bpermute(pull, (int)v.y);
        v.z = (uint32_t)__builtin_amdgcn_ds_bpermute(pull, (int)v.z);
        v.w = (uint32_t)__builtin_amdgcn_ds_bpermute(pull, (int)v.w);
    };
#pragma unroll
    for (int u = 0; u < N; ++u) {
        turn(x0[u]);
        turn(x1[u]);
    }
}

// Split `n_items` of one expert over `parts` workers: worker `sub` gets [first, last).
__device__ __forceinline__ void split_range(uint32_t n_items, uint32_t parts, uint32_t sub, uint32_t &first,
                                            uint32_t &last) {
    first = (uint32_t)((uint64_t)sub * n_items / parts);
    last = (uint32_t)((uint64_t)(sub + 1) * n_items / parts);
}

}  // namespace ffmoe
