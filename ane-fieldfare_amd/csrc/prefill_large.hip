// The prefill's two grouped products for layers that the fast forms do not hold.
#include "common.hpp"
#include "kernels.hpp"

namespace ffmoe {
namespace {

constexpr int kTilesPerBlock = 4;           // arena tiles (of 16 + 16 rows) of a block, a wave per tile

// Either product of a prefill chunk for a layer that has weight scales of 2^104 and more: 2^24 of them, which the GEMM's expansion
// and the FP16 form of the streaming product carry (prefill.hip), is infinite (and so is 128 of them from 2^121 on). Weights,
// tiles, layouts and the order of the sums are the GEMM's; the weights come by byte conversions and everything straight from
// memory. No model is known to have such a layer, so the time is not looked after: 3,072 rows of 128 experts of width 704 take
// 1.1 ms where the GEMMs take 0.34. A block has a set of four arena tiles, a wave per tile, against 64 pairs at a time.
template <bool GATE_UP, bool F16, bool DUMP>
__global__ __launch_bounds__(256) void prefill_large_scale_kernel(const uint8_t *__restrict__ arena_layer, ArenaGeom g,
                                                                  const PrefillPlan *__restrict__ plan,
                                                                  const PrefillTile *__restrict__ tiles,
                                                                  const uint32_t *__restrict__ sorted_token,
                                                                  const uint32_t *__restrict__ sorted_out_row,
                                                                  const uint16_t *__restrict__ a, uint32_t a_stride,
                                                                  uint16_t *__restrict__ out, uint32_t n_sets,
                                                                  float *__restrict__ act_scale, uint32_t act_blocks,
                                                                  uint4 *__restrict__ dump) {
    constexpr uint32_t kBlocks = 4;                         // 16-pair blocks at a time
    __shared__ float peaks[kTilesPerBlock][kBlocks * 16];
    const uint32_t set = blockIdx.x % n_sets, ti = blockIdx.x / n_sets;
    if (ti >= plan->n_tiles) return;
    const PrefillTile t = tiles[ti];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, j = lane & 15, jq = lane >> 4, tile = set * kTilesPerBlock + wave;
    const uint32_t n_groups = GATE_UP ? g.gd : g.gf, act_block0 = t.row_start / 16 + t.order;
    if (tile >= (GATE_UP ? g.gu_rb : g.dn_rbp)) return;     // (gate/up tiles make whole sets: its waves stay together)
    const uint8_t *expert = arena_layer + (size_t)t.expert * g.expert_bytes;
    const uint8_t *w_tiles = expert + (GATE_UP ? g.gu_tiles_off : g.dn_tiles_off) + (size_t)tile * n_groups * kTileBytes;
    const uint8_t *w_scales = expert + (GATE_UP ? g.gu_scales_off : g.dn_scales_off) + (size_t)tile * n_groups * kTileScaleBytes;
    for (uint32_t b0 = 0; b0 * 16 < t.rows; b0 += kBlocks) {
        f32x4 acc[kBlocks][2];
        const uint16_t *from[kBlocks];
#pragma unroll
        for (uint32_t m = 0; m < kBlocks; ++m) {
            const uint32_t block = min(b0 + m, (t.rows - 1) / 16);          // past the last the last again, never stored
            acc[m][0] = acc[m][1] = f32x4{0.f, 0.f, 0.f, 0.f};
            if constexpr (GATE_UP) from[m] = a + (size_t)sorted_token[t.row_start + min(block * 16 + j, t.rows - 1)] * a_stride + jq * 8;
            else from[m] = a + (size_t)(act_block0 + block) * n_groups * (2 * kWave * 8) + lane * 8;
        }
        for (uint32_t grp = 0; grp < n_groups; ++grp) {
            const uint4 w = reinterpret_cast<const uint4 *>(w_tiles + (size_t)grp * kTileBytes)[lane];
            const uint2 sc = reinterpret_cast<const uint2 *>(w_scales + (size_t)grp * kTileScaleBytes)[j];
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const uint4 weights[2] = {dequant8<F16>(half ? w.y : w.x, bf16lo_to_f32(sc.x), bf16hi_to_f32(sc.x)),
                                          dequant8<F16>(half ? w.w : w.z, bf16lo_to_f32(sc.y), bf16hi_to_f32(sc.y))};
#pragma unroll
                for (int st = 0; st < 2; ++st) {
                    if constexpr (DUMP) dump[(((size_t)set * n_groups + grp) * 16 + half * 8 + wave * 2 + st) * kWave + lane] = weights[st];
#pragma unroll
                    for (uint32_t m = 0; m < kBlocks; ++m) {
                        const uint4 x = *reinterpret_cast<const uint4 *>(from[m] + (GATE_UP ? grp * kGroup + half * 32 : (grp * 2 + half) * (kWave * 8)));
                        acc[m][st] = Act<F16>::mfma(weights[st], x, acc[m][st]);
                    }
                }
            }
        }
        // the epilogues of gemm_wave, without its detours through LDS
        if constexpr (GATE_UP) {
#pragma unroll
            for (uint32_t m = 0; m < kBlocks; ++m) {
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[m][0][r] = gelu_tanh_fast(acc[m][0][r]) * acc[m][1][r];
                if constexpr (F16) {
                    float peak = 0.0f;
#pragma unroll
                    for (int r = 0; r < 4; ++r) peak = fmaxf(peak, fabsf(acc[m][0][r]));
                    peak = fmaxf(peak, __shfl_xor(peak, 16, 64));
                    peak = fmaxf(peak, __shfl_xor(peak, 32, 64));
                    if (jq == 0) peaks[wave][16 * m + j] = peak;
                }
            }
            if constexpr (F16) __syncthreads();
#pragma unroll
            for (uint32_t m = 0; m < kBlocks; ++m) {
                const bool live = (b0 + m) * 16 + j < t.rows;
                if constexpr (F16) {
                    float peak = 0.0f;
#pragma unroll
                    for (int v = 0; v < kTilesPerBlock; ++v) peak = fmaxf(peak, peaks[v][16 * m + j]);
                    int e = 0;
                    (void)frexpf(peak, &e);
                    e = max(e, -100);
                    acc[m][0] *= ldexpf(1.0f, 14 - e);
                    if (live && jq == 0 && wave == 0) act_scale[((size_t)(act_block0 + b0 + m) * g.gf + set) * 16 + j] = ldexpf(1.0f, e - 14);
                }
                uint16_t *oblk = out + (((size_t)(act_block0 + b0 + m) * g.gf + set) * 2 + (tile >> 1 & 1)) * (kWave * 8);
                if (live)
                    *reinterpret_cast<uint2 *>(oblk + (((tile & 1) * 2 + (jq >> 1)) * 16 + j) * 8 + (jq & 1) * 4) =
                        make_uint2(Act<F16>::pack(acc[m][0][0], acc[m][0][1]), Act<F16>::pack(acc[m][0][2], acc[m][0][3]));
            }
            if constexpr (F16) __syncthreads();
        } else {
#pragma unroll
            for (uint32_t m = 0; m < kBlocks; ++m) {
                const uint32_t pair = (b0 + m) * 16 + j;
                if (pair >= t.rows) continue;
                float pair_largest = 1.0f;
                if constexpr (F16) pair_largest = act_scale[(size_t)act_blocks * g.gf * 16 + act_block0 * 16 + pair];
                uint16_t *row = out + (size_t)sorted_out_row[t.row_start + pair] * g.d + tile * (2 * kTileRows) + 4 * jq;
#pragma unroll
                for (int st = 0; st < 2; ++st) {
                    if constexpr (F16) acc[m][st] *= pair_largest;
                    *reinterpret_cast<uint2 *>(row + st * kTileRows) =
                        make_uint2(Act<F16>::pack(acc[m][st][0], acc[m][st][1]), Act<F16>::pack(acc[m][st][2], acc[m][st][3]));
                }
            }
        }
    }
}

}  // namespace

hipError_t launch_prefill_large_scale(hipStream_t s, const uint8_t *arena_layer, ArenaGeom g, bool gate_up, uint32_t tile_cap, const uint16_t *a,
                                      uint32_t a_stride, uint16_t *out, PrefillScratch sc, bool f16, void *dump) {
    const uint32_t sets = ((gate_up ? g.gu_rb : g.dn_rbp) + kTilesPerBlock - 1) / kTilesPerBlock;
    auto launch = [&](auto gate_up_, auto f16_, auto dump_) {
        hipLaunchKernelGGL((prefill_large_scale_kernel<decltype(gate_up_)::value, decltype(f16_)::value, decltype(dump_)::value>), dim3(tile_cap * sets), dim3(256),
                           0, s, arena_layer, g, sc.plan, sc.tiles, sc.sorted_token, sc.sorted_out_row, a, a_stride, out, sets, sc.act_scale,
                           sc.act_blocks, static_cast<uint4 *>(dump));
    };
    auto with_dump = [&](auto gate_up_, auto f16_) { dump ? launch(gate_up_, f16_, std::true_type{}) : launch(gate_up_, f16_, std::false_type{}); };
    auto with_type = [&](auto gate_up_) { f16 ? with_dump(gate_up_, std::true_type{}) : with_dump(gate_up_, std::false_type{}); };
    gate_up ? with_type(std::true_type{}) : with_type(std::false_type{});
    return hipGetLastError();
}

}  // namespace ffmoe
