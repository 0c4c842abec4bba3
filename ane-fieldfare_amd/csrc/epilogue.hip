// The steps either side of the MoE stage, one block per token row:
//   post-attention setup  fused_post_attn_setup (Metal/Fusions/fused.metal:210-296) and its block form
//                         prefill_post_attn_setup_block (Metal/Prefill/prefill.metal:243-318)
//   layer tail            prefill_layer_tail_block (Metal/Prefill/prefill.metal:320-399) and the decode
//                         tail of Kernels/Fusions/FusedLayerTail.swift
// Both are RMS norms around residual adds with every intermediate rounded to 16 bits where the reference
// rounds to FP16. A thread keeps its elements in registers from the first read to the last write (the
// reference stages rows in threadgroup memory); a row is read once and written once: HBM-bound.
// Every input row and every weight vector of a launch is requested before the first reduction, so a launch is one
// memory round trip and its block reductions (a load issued behind a reduction is another dependent round trip, and
// at 16 rows these kernels are nothing but their round trips); no value is converted before the last of a thread's requests
// is out (beside its load it was waited for, and the second chunk of a row went out a round trip later: setup of 1 row of 2,816 3.16 us, now
// 3.04; tail of 3,072 rows 16.0 | 15.5, of 8,192 33.1 | 31.3).
//
// Summation order of the squares (the reference's simd_sum leaves it open): thread t owns the 8-element
// chunks t, t + 256, ... and adds their squares in index order with fmaf; the wave meets in a
// xor-butterfly; the four wave sums combine as (w0 + w1) + (w2 + w3); inv = 1 / sqrt(sum / D + eps) with
// IEEE division and square root. Rows that are not 16-byte aligned take scalar loads of the same elements,
// so both paths give the same bits.
#include "common.hpp"
#include "kernels.hpp"

namespace ffmoe {
namespace {

constexpr int kRowThreads = 256;
constexpr int kMaxChunks = 2;        // D <= 4096: at most two 8-element chunks per thread
// Up to how many rows the tail converts before its first reduction: four of its blocks run on a compute unit then, two with the norms. us, late |
// early, 2,816 columns: 1 row 3.03 | 2.98, 100 rows 3.34 | 3.28, 301 rows 4.18 | 4.02, 1,000 rows 5.82 | 5.56 (3,072 rows 12.9 | 13.4); 4,096 columns, 1,000 rows
// 6.66 | 6.27; with the norms 301 rows 5.84 | 5.66, 500 rows 6.19 | 6.02 (1,000 rows 9.2 | 9.8, 8,192 rows 41 | 57).
constexpr uint32_t kEarlyRows = 1024, kEarlyNormRows = 512;

struct Row8 {
    float v[8];
};

// Rows are in the context's activation type (F16: FP16, else bf16); norm weights are always bf16.
template <bool VEC>
__device__ __forceinline__ uint4 load_raw8(const uint16_t *__restrict__ row, uint32_t chunk) {
    if (VEC) return reinterpret_cast<const uint4 *>(row)[chunk];
    const uint16_t *p = row + 8 * chunk;
    return make_uint4(p[0] | (uint32_t)p[1] << 16, p[2] | (uint32_t)p[3] << 16, p[4] | (uint32_t)p[5] << 16, p[6] | (uint32_t)p[7] << 16);
}

template <bool F16>
__device__ __forceinline__ Row8 widen8(const uint4 &q) {
    Row8 r;
    r.v[0] = Act<F16>::lo(q.x); r.v[1] = Act<F16>::hi(q.x);
    r.v[2] = Act<F16>::lo(q.y); r.v[3] = Act<F16>::hi(q.y);
    r.v[4] = Act<F16>::lo(q.z); r.v[5] = Act<F16>::hi(q.z);
    r.v[6] = Act<F16>::lo(q.w); r.v[7] = Act<F16>::hi(q.w);
    return r;
}

// A value on its way to 16 bits is an fp32 number first, as in the reference: left alone, the compiler makes a product and its rounding
// to FP16 one v_fma_mixlo_f16, which rounds once (some 5 of 100,000 values off by one bit).
template <bool F16>
__device__ __forceinline__ float as_f32(float x) {
    if (F16) asm("" : "+v"(x));
    return x;
}
template <bool F16>
__device__ __forceinline__ float round16(float x) { return Act<F16>::widen(Act<F16>::round(as_f32<F16>(x))); }

template <bool F16>
__device__ __forceinline__ uint4 pack8(const Row8 &r) {
    auto pair = [&](int e) { return Act<F16>::pack(as_f32<F16>(r.v[e]), as_f32<F16>(r.v[e + 1])); };
    return make_uint4(pair(0), pair(2), pair(4), pair(6));
}

template <bool VEC, bool F16>
__device__ __forceinline__ void store8(uint16_t *__restrict__ row, uint32_t chunk, const Row8 &r) {
    if (VEC) {
        reinterpret_cast<uint4 *>(row)[chunk] = pack8<F16>(r);
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) row[8 * chunk + e] = Act<F16>::round(as_f32<F16>(r.v[e]));
    }
}


// 1 / sqrt(mean of squares + eps) over the block's row; `slot` is a 4-float LDS area of its own
__device__ __forceinline__ float block_rms_inv(const Row8 (&x)[kMaxChunks], uint32_t n_mine, uint32_t d, float eps,
                                               float *slot) {
    float acc = 0.0f;
#pragma unroll
    for (int c = 0; c < kMaxChunks; ++c)
        if ((uint32_t)c < n_mine)
#pragma unroll
            for (int e = 0; e < 8; ++e) acc = __builtin_fmaf(x[c].v[e], x[c].v[e], acc);
    acc = wave_butterfly_sum(acc);
    if ((threadIdx.x & 63) == 0 && threadIdx.x < kRowThreads) slot[threadIdx.x >> 6] = acc;
    __syncthreads();
    const float total = (slot[0] + slot[1]) + (slot[2] + slot[3]);
    return 1.0f / sqrtf(total / (float)d + eps);
}

template <bool VEC, bool F16>
__global__ __launch_bounds__(kRowThreads) void post_attn_setup_kernel(
    uint16_t *__restrict__ hidden, const uint16_t *__restrict__ attn, const uint16_t *__restrict__ w_post_attn, uint32_t hidden_stride,
    uint32_t attn_stride, uint32_t d, float eps, const uint16_t *__restrict__ w_pre_ffn, const uint16_t *__restrict__ w_pre_ffn2,
    uint16_t *__restrict__ dense_x, uint16_t *__restrict__ routed_x, uint16_t *__restrict__ router_x, uint32_t dense_stride,
    uint32_t routed_stride, uint32_t router_stride) {
    __shared__ float s_sum[2][4];
    const uint32_t row = blockIdx.x, t = threadIdx.x, chunks = d / 8;
    const uint32_t n_mine = t < chunks ? (chunks - t + kRowThreads - 1) / kRowThreads : 0;
    uint16_t *hrow = hidden + (size_t)row * hidden_stride;
    const uint16_t *arow = attn + (size_t)row * attn_stride;
    uint4 a_raw[kMaxChunks], h_raw[kMaxChunks], w0_raw[kMaxChunks], w1_raw[kMaxChunks], w2_raw[kMaxChunks];
#pragma unroll
    for (int c = 0; c < kMaxChunks; ++c)
        if ((uint32_t)c < n_mine) {
            const uint32_t chunk = t + c * kRowThreads;
            a_raw[c] = load_raw8<VEC>(arow, chunk);
            h_raw[c] = load_raw8<VEC>(hrow, chunk);
            w0_raw[c] = load_raw8<VEC>(w_post_attn, chunk);
            w1_raw[c] = load_raw8<VEC>(w_pre_ffn, chunk);
            w2_raw[c] = load_raw8<VEC>(w_pre_ffn2, chunk);
        }
    Row8 a[kMaxChunks], h[kMaxChunks], w0[kMaxChunks], w1[kMaxChunks], w2[kMaxChunks];
#pragma unroll
    for (int c = 0; c < kMaxChunks; ++c) {
        a[c] = widen8<F16>(a_raw[c]);
        h[c] = widen8<F16>(h_raw[c]);
        w0[c] = widen8<false>(w0_raw[c]);
        w1[c] = widen8<false>(w1_raw[c]);
        w2[c] = widen8<false>(w2_raw[c]);
    }
    const float attn_inv = block_rms_inv(a, n_mine, d, eps, s_sum[0]);
#pragma unroll
    for (int c = 0; c < kMaxChunks; ++c)
        if ((uint32_t)c < n_mine) {
#pragma unroll
            for (int e = 0; e < 8; ++e) h[c].v[e] = round16<F16>(h[c].v[e] + round16<F16>(a[c].v[e] * attn_inv * w0[c].v[e]));
            store8<VEC, F16>(hrow, t + c * kRowThreads, h[c]);
        }
    const float hidden_inv = block_rms_inv(h, n_mine, d, eps, s_sum[1]);
#pragma unroll
    for (int c = 0; c < kMaxChunks; ++c)
        if ((uint32_t)c < n_mine) {
            const uint32_t chunk = t + c * kRowThreads;
            Row8 o_dense, o_routed, o_router;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float v = h[c].v[e] * hidden_inv;
                o_dense.v[e] = v * w1[c].v[e];
                o_routed.v[e] = v * w2[c].v[e];
                o_router.v[e] = v;
            }
            store8<VEC, F16>(dense_x + (size_t)row * dense_stride, chunk, o_dense);
            store8<VEC, F16>(routed_x + (size_t)row * routed_stride, chunk, o_routed);
            store8<VEC, F16>(router_x + (size_t)row * router_stride, chunk, o_router);
        }
}

// Where h2 comes from when the routed experts' rows arrive un-combined (COMBINE): the un-weighted fp32 rows of a
// decode / verify call, the routes' weights and the plan's validity words. h2 = the combine kernel's row: fmaf over
// the valid routes in rank order from zero, one rounding to 16 bits - made in this kernel's load stage instead of a
// launch of its own, with the same arithmetic, so the tail's results keep their bits.
struct RoutedRows {
    const float *partials;           // [t * top_k][d]
    const uint16_t *w;               // [t][top_k]
    const uint32_t *route_valid;     // [t * top_k]
    uint32_t top_k;
    // h1 likewise, when the shared expert's down projection rode along in the routed experts' launch and left its K in
    // chunks: h1 = the chunks' fp32 rows added in chunk order, one rounding to 16 bits (what the dense FFN's own down
    // launch rounds once too). Null: h1 is read as a 16-bit row.
    const float *shared_partials;    // [shared_chunks][t][d]
    uint32_t shared_chunks, t;
};

// What a chunk of h2 (and of h1) is made of. The routes' weights and validity words come as one load each, a route per lane: read
// where they are wanted, route after route, the words were eight scalar loads one behind the other.
struct RoutedChunk {
    f32x4 lo[8], hi[8], shared_lo[4], shared_hi[4];
};

__device__ __forceinline__ RoutedChunk load_routed(const RoutedRows &rr, uint32_t row, uint32_t d, uint32_t chunk) {
    RoutedChunk in;
#pragma unroll
    for (uint32_t r = 0; r < 8; ++r) {
        const float *src = rr.partials + (size_t)(row * rr.top_k + min(r, rr.top_k - 1)) * d + 8 * chunk;
        in.lo[r] = *reinterpret_cast<const f32x4 *>(src);
        in.hi[r] = *reinterpret_cast<const f32x4 *>(src + 4);
    }
    if (rr.shared_partials)
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) {
            const float *src = rr.shared_partials + ((size_t)min(c, rr.shared_chunks - 1) * rr.t + row) * d + 8 * chunk;
            in.shared_lo[c] = *reinterpret_cast<const f32x4 *>(src);
            in.shared_hi[c] = *reinterpret_cast<const f32x4 *>(src + 4);
        }
    return in;
}

template <bool F16>
__device__ __forceinline__ Row8 shared_row8(const RoutedRows &rr, const RoutedChunk &in) {
    Row8 out;
#pragma unroll
    for (int i = 0; i < 8; ++i) out.v[i] = 0.0f;
#pragma unroll
    for (uint32_t c = 0; c < 4; ++c) {
        if (c < rr.shared_chunks) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                out.v[i] += in.shared_lo[c][i];
                out.v[4 + i] += in.shared_hi[c][i];
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) out.v[i] = round16<F16>(out.v[i]);
    return out;
}

// lane r: route r's weight bits and validity word (also where lane r itself has no chunk)
template <bool F16>
__device__ __forceinline__ Row8 combine8(const RoutedChunk &in, uint32_t top_k, uint32_t weight, uint32_t valid) {
    Row8 out;
#pragma unroll
    for (int i = 0; i < 8; ++i) out.v[i] = 0.0f;
#pragma unroll
    for (uint32_t r = 0; r < 8; ++r) {
        const float wv = Act<F16>::widen((uint16_t)__builtin_amdgcn_readlane((int)weight, (int)r));
        if (r < top_k && __builtin_amdgcn_readlane((int)valid, (int)r) != 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                out.v[i] = __builtin_fmaf(wv, in.lo[r][i], out.v[i]);
                out.v[4 + i] = __builtin_fmaf(wv, in.hi[r][i], out.v[4 + i]);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) out.v[i] = round16<F16>(out.v[i]);
    return out;
}

// NORMS: h1 arrives before its own norm (w_postffn1) and, when w_next is given, the norm of the new hidden
// row under w_next goes to `normed` (the next layer's input norm): fused_layer_tail_norms
// (Kernels/Fusions/FusedLayerTail.swift:74-117). h1 itself is left as it was found.
// COMBINE: rows of more than 256 chunks have a thread per chunk for the combining, which is 24 loads of 16 bytes for one: those past the
// 256th hand their chunks, rounded to 16 bits as they are, to the threads that own them in the order of the sums. 1 row of
// 2,816, us per launch: both chunks by their owner, each behind its own chain of loads 5.9, so 4.6.
// EARLY: a thread's chunks are fp32 numbers, and only where it has them, before the first reduction, in 123 registers (171 with NORMS); else they stay
// as they came, in 62 (74), and are converted behind each. The first is the shorter chain, the second more blocks per compute unit: kEarlyRows.
template <bool VEC, bool NORMS, bool F16, bool COMBINE = false, bool EARLY = false>
__global__ __launch_bounds__(COMBINE ? 2 * kRowThreads : kRowThreads) void layer_tail_kernel(const uint16_t *__restrict__ h1, uint16_t *__restrict__ hidden,
                                                                 const uint16_t *__restrict__ w_postffn2,
                                                                 const uint16_t *__restrict__ w_postffn,
                                                                 const uint16_t *__restrict__ h2, uint32_t h2_stride, uint32_t h1_stride,
                                                                 uint32_t hidden_stride, uint32_t d, float eps, float layer_scalar,
                                                                 const uint16_t *__restrict__ w_postffn1,
                                                                 const uint16_t *__restrict__ w_next,
                                                                 uint16_t *__restrict__ normed, uint32_t normed_stride,
                                                                 RoutedRows routed) {
    __shared__ float s_sum[4][4];
    const uint32_t row = blockIdx.x, t = threadIdx.x, chunks = d / 8;
    const uint32_t n_mine = t < min(chunks, (uint32_t)kRowThreads) ? (chunks - t + kRowThreads - 1) / kRowThreads : 0;
    uint16_t *hrow = hidden + (size_t)row * hidden_stride;
    Row8 a[kMaxChunks], h12[kMaxChunks], hv[kMaxChunks], wf1[kMaxChunks], wf2[kMaxChunks], wf[kMaxChunks], wn[kMaxChunks];
    if constexpr (COMBINE) {
        // every load before the first use of one: converted beside their loads, a thread's chunks were a round trip each
        __shared__ uint4 handed[2][kRowThreads];        // h2, h1: chunks 256 .. 511
        const bool h1_given = !routed.shared_partials;
        uint4 h1_raw[kMaxChunks], h_raw[kMaxChunks], wf2_raw[kMaxChunks], wf_raw[kMaxChunks];
#pragma unroll
        for (int c = 0; c < kMaxChunks; ++c)
            if ((uint32_t)c < n_mine) {
                const uint32_t chunk = t + c * kRowThreads;
                if (h1_given) h1_raw[c] = load_raw8<VEC>(h1 + (size_t)row * h1_stride, chunk);
                h_raw[c] = load_raw8<VEC>(hrow, chunk);
                wf2_raw[c] = load_raw8<VEC>(w_postffn2, chunk);
                wf_raw[c] = load_raw8<VEC>(w_postffn, chunk);
            }
        const uint32_t route = row * routed.top_k + min(t & 63, routed.top_k - 1);
        const uint32_t weight = routed.w[route], valid = routed.route_valid[route];
        uint4 h2_raw = {0, 0, 0, 0};
        if (t < chunks) {
            const RoutedChunk in = load_routed(routed, row, d, t);
            h2_raw = pack8<F16>(combine8<F16>(in, routed.top_k, weight, valid));
            uint4 h1_mine = {0, 0, 0, 0};
            if (!h1_given) h1_mine = pack8<F16>(shared_row8<F16>(routed, in));
            if (t < kRowThreads) {
                if (!h1_given) h1_raw[0] = h1_mine;
            } else {
                handed[0][t - kRowThreads] = h2_raw;
                handed[1][t - kRowThreads] = h1_mine;
            }
        }
        __syncthreads();
        if (n_mine > 1) {
            a[1] = widen8<F16>(handed[0][t]);
            if (!h1_given) h1_raw[1] = handed[1][t];
        }
        a[0] = widen8<F16>(h2_raw);
#pragma unroll
        for (int c = 0; c < kMaxChunks; ++c) {
            h12[c] = widen8<F16>(h1_raw[c]);
            hv[c] = widen8<F16>(h_raw[c]);
            wf2[c] = widen8<false>(wf2_raw[c]);
            wf[c] = widen8<false>(wf_raw[c]);
        }
    } else {
        uint4 a_raw[kMaxChunks], h1_raw[kMaxChunks], h_raw[kMaxChunks], wf2_raw[kMaxChunks], wf_raw[kMaxChunks], wf1_raw[kMaxChunks], wn_raw[kMaxChunks];
#pragma unroll
        for (int c = 0; c < kMaxChunks; ++c)
            if ((uint32_t)c < n_mine) {
                const uint32_t chunk = t + c * kRowThreads;
                a_raw[c] = load_raw8<VEC>(h2 + (size_t)row * h2_stride, chunk);
                h1_raw[c] = load_raw8<VEC>(h1 + (size_t)row * h1_stride, chunk);
                h_raw[c] = load_raw8<VEC>(hrow, chunk);
                wf2_raw[c] = load_raw8<VEC>(w_postffn2, chunk);
                wf_raw[c] = load_raw8<VEC>(w_postffn, chunk);
                if (NORMS) wf1_raw[c] = load_raw8<VEC>(w_postffn1, chunk);
                if (NORMS) wn_raw[c] = load_raw8<VEC>(w_next ? w_next : w_postffn1, chunk);
            }
#pragma unroll
        for (int c = 0; c < kMaxChunks; ++c) {
            if (EARLY && (uint32_t)c >= n_mine) break;
            a[c] = widen8<F16>(a_raw[c]);
            h12[c] = widen8<F16>(h1_raw[c]);
            hv[c] = widen8<F16>(h_raw[c]);
            wf2[c] = widen8<false>(wf2_raw[c]);
            wf[c] = widen8<false>(wf_raw[c]);
            if (NORMS) wf1[c] = widen8<false>(wf1_raw[c]);
            if (NORMS) wn[c] = widen8<false>(wn_raw[c]);
        }
    }
    if (NORMS) {
        const float inv_h1 = block_rms_inv(h12, n_mine, d, eps, s_sum[2]);
#pragma unroll
        for (int c = 0; c < kMaxChunks; ++c)
            if ((uint32_t)c < n_mine) {
#pragma unroll
                for (int e = 0; e < 8; ++e) h12[c].v[e] = round16<F16>(h12[c].v[e] * inv_h1 * wf1[c].v[e]);
            }
    }
    const float inv_h2 = block_rms_inv(a, n_mine, d, eps, s_sum[0]);
#pragma unroll
    for (int c = 0; c < kMaxChunks; ++c)
        if ((uint32_t)c < n_mine) {
#pragma unroll
            for (int e = 0; e < 8; ++e) h12[c].v[e] = round16<F16>(h12[c].v[e] + round16<F16>(a[c].v[e] * inv_h2 * wf2[c].v[e]));
        }
    const float inv_h12 = block_rms_inv(h12, n_mine, d, eps, s_sum[1]);
    const float scale = round16<F16>(layer_scalar);
#pragma unroll
    for (int c = 0; c < kMaxChunks; ++c)
        if ((uint32_t)c < n_mine) {
            const uint32_t chunk = t + c * kRowThreads;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                hv[c].v[e] = round16<F16>(round16<F16>(hv[c].v[e] + round16<F16>(h12[c].v[e] * inv_h12 * wf[c].v[e])) * scale);
            store8<VEC, F16>(hrow, chunk, hv[c]);
            a[c] = hv[c];          // the new hidden row, as stored
        }
    if (NORMS && w_next) {
        const float inv_next = block_rms_inv(a, n_mine, d, eps, s_sum[3]);
#pragma unroll
        for (int c = 0; c < kMaxChunks; ++c)
            if ((uint32_t)c < n_mine) {
                const uint32_t chunk = t + c * kRowThreads;
                const Row8 &w = wn[c];
                Row8 o;
#pragma unroll
                for (int e = 0; e < 8; ++e) o.v[e] = a[c].v[e] * inv_next * w.v[e];
                store8<VEC, F16>(normed + (size_t)row * normed_stride, chunk, o);
            }
    }
}

// rmsnorm_bf16w (RMSNorm.encodeBF16W): out = round((x * inv) * w) per row; out may be x.
template <bool VEC, bool F16>
__global__ __launch_bounds__(kRowThreads) void rmsnorm_kernel(const uint16_t *x, uint32_t x_stride, const uint16_t *__restrict__ w,
                                                              uint16_t *out, uint32_t out_stride, uint32_t d, float eps) {
    __shared__ float s_sum[4];
    const uint32_t row = blockIdx.x, t = threadIdx.x, chunks = d / 8;
    const uint32_t n_mine = t < chunks ? (chunks - t + kRowThreads - 1) / kRowThreads : 0;
    uint4 a_raw[kMaxChunks], w_raw[kMaxChunks];
#pragma unroll
    for (int c = 0; c < kMaxChunks; ++c)
        if ((uint32_t)c < n_mine) {
            a_raw[c] = load_raw8<VEC>(x + (size_t)row * x_stride, t + c * kRowThreads);
            w_raw[c] = load_raw8<VEC>(w, t + c * kRowThreads);
        }
    Row8 a[kMaxChunks], wq[kMaxChunks];
#pragma unroll
    for (int c = 0; c < kMaxChunks; ++c) {
        if ((uint32_t)c >= n_mine) break;       // (early: 51 registers, eight waves per SIMD either way; 1,000 rows of 2,816 3.48 -> 3.36 us)
        a[c] = widen8<F16>(a_raw[c]);
        wq[c] = widen8<false>(w_raw[c]);
    }
    const float inv = block_rms_inv(a, n_mine, d, eps, s_sum);
#pragma unroll
    for (int c = 0; c < kMaxChunks; ++c)
        if ((uint32_t)c < n_mine) {
            const uint32_t chunk = t + c * kRowThreads;
            const Row8 &wv = wq[c];
            Row8 o;
#pragma unroll
            for (int e = 0; e < 8; ++e) o.v[e] = a[c].v[e] * inv * wv.v[e];
            store8<VEC, F16>(out + (size_t)row * out_stride, chunk, o);
        }
}

bool aligned16(const void *p, uint32_t stride) { return reinterpret_cast<uintptr_t>(p) % 16 == 0 && stride % 8 == 0; }

}  // namespace

hipError_t launch_post_attn_setup(hipStream_t s, uint16_t *hidden, uint32_t hidden_stride, const uint16_t *attn,
                                  uint32_t attn_stride, uint16_t *dense_x, uint32_t dense_stride, uint16_t *routed_x,
                                  uint32_t routed_stride, uint16_t *router_x, uint32_t router_stride,
                                  const uint16_t *w_post_attn, const uint16_t *w_pre_ffn, const uint16_t *w_pre_ffn2,
                                  uint32_t t, uint32_t d, float eps, bool f16) {
    const bool vec = aligned16(hidden, hidden_stride) && aligned16(attn, attn_stride) && aligned16(dense_x, dense_stride) &&
                     aligned16(routed_x, routed_stride) && aligned16(router_x, router_stride) && aligned16(w_post_attn, 8) &&
                     aligned16(w_pre_ffn, 8) && aligned16(w_pre_ffn2, 8);
#define FFMOE_SETUP(V, H)                                                                                                  \
    hipLaunchKernelGGL((post_attn_setup_kernel<V, H>), dim3(t), dim3(kRowThreads), 0, s, hidden, attn, w_post_attn, hidden_stride, attn_stride, \
                       d, eps, w_pre_ffn, w_pre_ffn2, dense_x, routed_x, router_x, dense_stride, routed_stride, router_stride)
    if (f16) { if (vec) FFMOE_SETUP(true, true); else FFMOE_SETUP(false, true); }
    else { if (vec) FFMOE_SETUP(true, false); else FFMOE_SETUP(false, false); }
#undef FFMOE_SETUP
    return hipGetLastError();
}

hipError_t launch_layer_tail(hipStream_t s, const uint16_t *h2, uint32_t h2_stride, const uint16_t *h1, uint32_t h1_stride,
                             uint16_t *hidden, uint32_t hidden_stride, const uint16_t *w_postffn2, const uint16_t *w_postffn,
                             uint32_t t, uint32_t d, float eps, float layer_scalar, const uint16_t *w_postffn1,
                             const uint16_t *w_next, uint16_t *normed, uint32_t normed_stride, bool f16,
                             const float *routed_partials, const uint16_t *routed_w, const uint32_t *route_valid, uint32_t top_k,
                             const float *shared_partials, uint32_t shared_chunks) {
    const bool norms = w_postffn1 != nullptr;
    if (shared_partials && (!routed_partials || shared_chunks == 0 || shared_chunks > 4)) return hipErrorInvalidValue;
    const RoutedRows routed{routed_partials, routed_w, route_valid, top_k, shared_partials, shared_chunks, t};
    if (routed_partials) {
        // h2 is made from the un-combined rows (16-byte aligned fp32 rows: d % 8 == 0); the plain tail only
        const bool vec = (shared_partials || aligned16(h1, h1_stride)) && aligned16(hidden, hidden_stride) && aligned16(w_postffn2, 8) && aligned16(w_postffn, 8);
#define FFMOE_TAILC(V, H)                                                                                             \
    hipLaunchKernelGGL((layer_tail_kernel<V, false, H, true>), dim3(t), dim3(d / 8 > kRowThreads ? 2 * kRowThreads : kRowThreads), 0, s, h1, hidden, \
                       w_postffn2, w_postffn, nullptr, 0u, h1_stride, hidden_stride, d, eps, layer_scalar, nullptr, nullptr, nullptr, 0u, routed)
        if (f16) { if (vec) FFMOE_TAILC(true, true); else FFMOE_TAILC(false, true); }
        else { if (vec) FFMOE_TAILC(true, false); else FFMOE_TAILC(false, false); }
#undef FFMOE_TAILC
        return hipGetLastError();
    }
    const bool vec = aligned16(h2, h2_stride) && aligned16(h1, h1_stride) && aligned16(hidden, hidden_stride) &&
                     aligned16(w_postffn2, 8) && aligned16(w_postffn, 8) &&
                     (!norms || (aligned16(w_postffn1, 8) && (!w_next || (aligned16(w_next, 8) && aligned16(normed, normed_stride)))));
    // (as many rows as blocks of the early form that run at once)
    const bool early = t <= (norms ? kEarlyNormRows : kEarlyRows);
#define FFMOE_TAIL_AS(V, N, H, E)                                                                                     \
    hipLaunchKernelGGL((layer_tail_kernel<V, N, H, false, E>), dim3(t), dim3(kRowThreads), 0, s, h1, hidden, w_postffn2, \
                       w_postffn, h2, h2_stride, h1_stride, hidden_stride, d, eps, layer_scalar, w_postffn1, w_next, normed, \
                       normed_stride, routed)
#define FFMOE_TAIL(V, N)                                                                                              \
    do {                                                                                                              \
        if (f16) { if (early) FFMOE_TAIL_AS(V, N, true, true); else FFMOE_TAIL_AS(V, N, true, false); }               \
        else { if (early) FFMOE_TAIL_AS(V, N, false, true); else FFMOE_TAIL_AS(V, N, false, false); }                 \
    } while (0)
    if (vec) { if (norms) FFMOE_TAIL(true, true); else FFMOE_TAIL(true, false); }
    else { if (norms) FFMOE_TAIL(false, true); else FFMOE_TAIL(false, false); }
#undef FFMOE_TAIL
#undef FFMOE_TAIL_AS
    return hipGetLastError();
}

hipError_t launch_rmsnorm(hipStream_t s, const uint16_t *x, uint32_t x_stride, const uint16_t *w, uint16_t *out,
                          uint32_t out_stride, uint32_t t, uint32_t d, float eps, bool f16) {
    const bool vec = aligned16(x, x_stride) && aligned16(out, out_stride) && aligned16(w, 8);
#define FFMOE_NORM(V, H) \
    hipLaunchKernelGGL((rmsnorm_kernel<V, H>), dim3(t), dim3(kRowThreads), 0, s, x, x_stride, w, out, out_stride, d, eps)
    if (f16) { if (vec) FFMOE_NORM(true, true); else FFMOE_NORM(false, true); }
    else { if (vec) FFMOE_NORM(true, false); else FFMOE_NORM(false, false); }
#undef FFMOE_NORM
    return hipGetLastError();
}

}  // namespace ffmoe
