"""The work that a program serving a Gemma-4-26B-A4B-shaped model gives this library, one case per call pattern, over the
sizes it meets: hidden 2,816, 128 routed experts of width 704 with top-8 routing, a shared expert of width 2,112 and a head
of 262,144 rows, all INT4 (the shared expert also 8-bit, the form in which the model's packs hold it). Everything goes
through the Python binding, as a program's own loop would.

Kinds of case:
  projection  one resident INT4 matrix on the 1 to 16 rows of a step (the attention projections of a layer)
  block       a layer's whole MoE block for the 1 to 16 rows of a decode step or a verify block: embedding rows into the
              residual stream, post-attention setup, router + routed experts + shared expert in one call, layer tail
  verify      router + routed experts + residual alone for such a block
  prompt      the same layer block for a prompt or a chunk of one, 17 rows up: router, prefill, dense FFN as calls of their
              own; with `zipf` the routes are given and skewed as a topic skews them (no router call)
  guest       the plugin contract for a prefill chunk: expert-sorted pairs in, un-weighted rows out, then the reduce
  greedy      the head's choice and its confidence for each row of a step
  sample      the head's logits and a draw from their tempered, truncated softmax
  hot         the drafter's guess over a list of frequent tokens: listed rows of the table, then the choice among them
"""
import math
import os
import sys

_PACKAGE = os.path.join(os.getcwd(), "ane-fieldfare_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(1, _PACKAGE)

import numpy as np
import torch

import fieldfare_moe as ff
from fieldfare_moe import synthetic as syn

D, F, E, K, VOCAB = syn.D, syn.F, syn.E, syn.K, syn.VOCAB
SHARED_F = 2112
CHUNK = 4096            # the longest prompt chunk a context is made for, unless a case needs more
EXPERT_BYTES = syn.EXPERT_BYTES


def listed():
    return [
        # the smallest call there is: one attention-sized projection for one decoded token; a launch and little else
        {"name": "projection_1row", "kind": "projection", "rows": 1, "m": 1408, "n": 2816, "dtype": "bf16"},
        # a decode step's layer: one token, the packs' default shared expert; the latency chain of plain decoding
        {"name": "block_1row", "kind": "block", "rows": 1, "shared_bits": 8, "dtype": "bf16"},
        # a short speculative block in the reference's text-path type, 4-bit shared expert; an odd row count
        {"name": "block_5rows_fp16", "kind": "block", "rows": 5, "shared_bits": 4, "dtype": "fp16"},
        # the 16-token verify block through the routed experts: about 50 distinct experts, the headline workload
        {"name": "verify_16rows", "kind": "verify", "rows": 16, "dtype": "bf16"},
        # a short chat turn: too long for one verify block, far too short to fill a grouped GEMM's tiles
        {"name": "prompt_37", "kind": "prompt", "rows": 37, "shared_bits": 8, "zipf": False, "dtype": "bf16"},
        # an ordinary question with a little context; every expert live, about 19 rows each
        {"name": "prompt_301", "kind": "prompt", "rows": 301, "shared_bits": 4, "zipf": False, "dtype": "bf16"},
        # the plugin boundary at a middling chunk, FP16 as the reference's host hands it over
        {"name": "guest_1000_fp16", "kind": "guest", "rows": 1000, "dtype": "fp16"},
        # the long-prompt chunk the prefill half of the headline is quoted on
        {"name": "prompt_3072", "kind": "prompt", "rows": 3072, "shared_bits": 8, "zipf": False, "dtype": "bf16"},
        # the largest chunk, with the skewed expert popularity of a single-topic document
        {"name": "prompt_8192_zipf", "kind": "prompt", "rows": 8192, "shared_bits": 4, "zipf": True, "dtype": "bf16"},
        # the head at the end of a verify block: choice and confidence of all sixteen rows
        {"name": "greedy_16rows", "kind": "greedy", "rows": 16, "dtype": "bf16"},
        # the head at the end of a sampled decode step, truncated as chat settings have it
        {"name": "sample_1row", "kind": "sample", "rows": 1, "top_k": 64, "top_p": 0.9, "temperature": 0.8, "dtype": "bf16"},
        # the drafter's hot vocabulary for a block of rows; 4,099 is the head size the reference's own head tests use
        {"name": "hot_4099_16rows", "kind": "hot", "rows": 16, "count": 4099, "dtype": "bf16"},
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(("projection", "block", "block", "verify", "prompt", "prompt", "prompt", "guest", "greedy", "sample", "hot"))
    case = {"kind": kind, "dtype": rng.choice(("bf16", "bf16", "fp16"))}
    if kind == "projection":
        # from a small head-sized projection to a wide fused one; any row count of the matrix, any group count of its columns
        case.update(rows=rng.randint(1, 16), m=_log_int(rng, 256, 16384), n=64 * rng.randint(8, 44))
    elif kind == "block":
        case.update(rows=rng.randint(1, 16), shared_bits=rng.choice((4, 8)))
    elif kind == "verify":
        case.update(rows=rng.randint(1, 16))
    elif kind == "prompt":
        case.update(rows=_log_int(rng, 17, 8192), shared_bits=rng.choice((4, 8)), zipf=rng.random() < 0.3)
        if case["rows"] > 4096:
            case.update(shared_bits=4)      # an 8-bit shared expert at these sizes would cost more than the largest listed case
            case.update(dtype="bf16")       # and so would FP16
    elif kind == "guest":
        case.update(rows=_log_int(rng, 17, 4096))
    elif kind == "greedy":
        case.update(rows=rng.randint(1, 16))
    elif kind == "sample":
        truncated = rng.random() < 0.7
        case.update(rows=rng.randint(1, 16), top_k=rng.randint(8, 256) if truncated else 0,
                    top_p=round(rng.uniform(0.8, 1.0), 2) if truncated else 1.0, temperature=round(rng.uniform(0.5, 1.3), 2))
    else:
        case.update(rows=rng.randint(1, 16), count=_log_int(rng, 512, 32768))
    return case


class _State:
    """A case's inputs and the handles a program keeps between calls."""


def _normal(gen, *shape):
    return torch.randn(shape, device="cuda", generator=gen)


def _affine8(gen, rows, cols):
    """An 8-bit affine weight in the packs' layout, with bytes around a zero point of 128."""
    w = torch.randint(0, 256, (rows, cols), dtype=torch.uint8, device="cuda", generator=gen)
    s = (_normal(gen, rows, cols // ff.GROUP) * 0.001).abs().to(torch.bfloat16)
    b = (-128.0 * s.float() + _normal(gen, rows, cols // ff.GROUP) * 1e-3).to(torch.bfloat16)
    return w, s, b


def _routed_context(gen, case, max_tokens):
    ctx = ff.Context(D, F, E, K, n_layers=1, max_tokens=max_tokens, act_dtype=case["dtype"])
    offsets, _ = syn.layout_offsets(D, F, align=16)
    ctx.upload_layer(0, syn.synth_layer_gpu(torch, gen, offsets).view(-1), syn.STRIDE, offsets)
    router = (_normal(gen, E, D) * 0.02).to(torch.bfloat16)
    ctx.upload_router_bf16(0, router.view(torch.int16).cpu().numpy().view(np.uint16))
    return ctx


def _shared_context(gen, case, max_tokens):
    ctx = ff.Context(D, SHARED_F, 1, 1, n_layers=1, max_tokens=max_tokens, act_dtype=case["dtype"])
    make = _affine8 if case["shared_bits"] == 8 else lambda g, rows, cols: syn.synth_matrix_gpu(torch, g, rows, cols)
    parts = [make(gen, rows, cols) for rows, cols in ((SHARED_F, D), (SHARED_F, D), (D, SHARED_F))]
    ctx.upload_expert_parts(0, 0, *parts, int8=case["shared_bits"] == 8)
    return ctx


def _zipf_routes(gen, rows, act):
    """top-8 distinct experts per token under Zipf(1.1) popularity (a Gumbel draw without replacement), weights that add to 1."""
    p = 1.0 / torch.arange(1, E + 1, device="cuda", dtype=torch.float32) ** 1.1
    popularity = (p / p.sum())[torch.randperm(E, device="cuda", generator=gen)]
    noise = -torch.log(-torch.log(torch.rand((rows, E), device="cuda", generator=gen).clamp(1e-9, 1 - 1e-7)))
    idx = torch.topk(popularity.log() + noise, K, dim=1).indices.to(torch.int32).contiguous()
    w = torch.rand((rows, K), device="cuda", generator=gen) + 0.05
    return idx, (w / w.sum(1, keepdim=True)).to(act)


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    s = _State()
    s.case, kind, rows = case, case["kind"], case["rows"]
    act = torch.bfloat16 if case["dtype"] == "bf16" else torch.float16
    if kind in ("projection", "greedy", "sample", "hot"):
        s.ctx = ff.Context(256, 128, 8, 8, n_layers=1, max_tokens=16, act_dtype=case["dtype"])
        n = case.get("n", D)
        weight = syn.synth_matrix_gpu(torch, gen, case.get("m", VOCAB), n)
        s.x = _normal(gen, rows, n).to(act)
        if kind == "hot":
            # the table in the reference's layout and the ids of the frequent tokens, in the order the list has them
            s.table = weight
            s.ids = torch.randperm(VOCAB, device="cuda", generator=gen)[:case["count"]].to(torch.int32)
        else:
            s.matrix = s.ctx.matrix(*weight, greedy=kind == "greedy")
        s.seed = seed
        return s
    max_tokens = max(CHUNK, rows)
    s.ctx = _routed_context(gen, case, max_tokens)
    if kind == "verify":
        s.x = syn.TOKEN_CORRELATION ** 0.5 * _normal(gen, 1, D) + (1 - syn.TOKEN_CORRELATION) ** 0.5 * _normal(gen, rows, D)
        s.x = s.x.to(act)
        s.residual = _normal(gen, rows, D).to(act)
        return s
    if kind == "guest":
        s.x = _normal(gen, rows, D).to(act)
        idx, s.w = s.ctx.router(0, s.x)
        order = torch.argsort(idx.reshape(-1), stable=True)
        s.pairs = torch.stack((order // K, idx.reshape(-1)[order].to(torch.int64), order % K,
                               s.w.reshape(-1)[order].view(torch.int16).to(torch.int64) & 0xFFFF), 1).to(torch.int32).contiguous()
        s.partials = torch.zeros((rows, K, D), dtype=act, device="cuda")
        return s
    s.shared = _shared_context(gen, case, max_tokens)
    # the tied table: the rows of a step's or a chunk's tokens enter the residual stream scaled by sqrt(hidden), about unit size
    table = [a if i == 0 else (a.float() * 0.4).to(torch.bfloat16) for i, a in enumerate(syn.synth_matrix_gpu(torch, gen, VOCAB))]
    s.table = s.ctx.matrix(*table)
    s.tokens = torch.randint(0, VOCAB, (rows,), dtype=torch.int32, device="cuda", generator=gen)
    # what attention returns for neighbouring tokens of a block has much in common: it is what makes a verify block's rows share experts
    common = 0.9 if kind == "block" else 0.0
    s.attn = (common ** 0.5 * _normal(gen, 1, D) + (1 - common) ** 0.5 * _normal(gen, rows, D)).to(act)
    s.norms = [(torch.rand((D,), device="cuda", generator=gen) + 0.5).to(torch.bfloat16) for _ in range(5)]
    s.hidden = torch.empty((rows, D), dtype=act, device="cuda")
    s.routes = _zipf_routes(gen, rows, act) if case.get("zipf") else None
    return s


def run(s):
    case, kind, ctx = s.case, s.case["kind"], s.ctx
    if kind == "projection":
        return s.matrix.gemv(s.x)
    if kind == "greedy":
        return s.matrix.greedy_conf(s.x, softcap=30.0)
    if kind == "sample":
        logits = s.matrix.gemv(s.x, f32_out=True)
        return (logits,) + ctx.sample_rows(logits, case["temperature"], 30.0, s.seed, key_base=100, top_k=case["top_k"],
                                           top_p=case["top_p"])
    if kind == "hot":
        logits = ctx.gemv_int4_listed(*s.table, s.ids, s.x)
        return (logits,) + ctx.argmax_rows(logits, softcap=30.0)
    if kind == "verify":
        return ctx.route_verify(0, s.x, s.x, residual=s.residual)
    if kind == "guest":
        ctx.prefill_pairs(0, s.x, s.pairs, case["rows"], s.partials)
        return s.partials, ctx.reduce_token_major(s.partials, s.w)
    s.table.rows(s.tokens, math.sqrt(D), out=s.hidden)
    dense_x, routed_x, router_x = ctx.post_attn_setup(s.hidden, s.attn, s.norms[0], s.norms[1], s.norms[2])
    if kind == "block":
        idx, w = ctx.route_verify_shared(s.shared, 0, 0, router_x, routed_x, dense_x)
        ctx.layer_tail_routed_shared(s.shared, w, s.hidden, s.norms[3], s.norms[4], 0.5)
        return s.hidden, idx, w
    idx, w = s.routes if s.routes is not None else ctx.router(0, router_x)
    h2 = ctx.prefill(0, routed_x, idx, w)
    h1 = s.shared.dense_ffn(0, dense_x)
    ctx.layer_tail(h2, h1, s.hidden, s.norms[3], s.norms[4], 0.5)
    return s.hidden, h2, h1, idx, w


def _matrix_bytes(m, n, bits=4):
    return m * n * bits / 8 + 4 * m * (n / ff.GROUP)


def _live_experts(case):
    """Distinct experts the rows reach: independent rows for prompts, fewer for a block whose rows have much in common (about 50
    for sixteen rows); under Zipf popularity every expert is met soon."""
    rows = case["rows"] ** 0.734 if case["kind"] in ("block", "verify") else case["rows"]
    return E * (1 - (1 - K / E) ** rows)


def work(case):
    kind, rows = case["kind"], case["rows"]
    row = 2 * D
    if kind == "projection":
        m, n = case["m"], case["n"]
        return {"bytes": _matrix_bytes(m, n) + 2 * rows * (m + n), "flops": 2.0 * rows * m * n}
    if kind in ("greedy", "sample"):
        logits = 4 * rows * VOCAB if kind == "sample" else 0
        return {"bytes": _matrix_bytes(VOCAB, D) + rows * row + logits, "flops": 2.0 * rows * VOCAB * D}
    if kind == "hot":
        count = case["count"]
        return {"bytes": _matrix_bytes(count, D) + 4 * count + rows * row + 4 * rows * count, "flops": 2.0 * rows * count * D}
    experts = _live_experts(case) * EXPERT_BYTES
    flops = 2.0 * rows * K * 3 * D * F
    if kind == "guest":
        # pairs, rows and experts read, the un-weighted rows written, read by the reduce, the combined rows written
        return {"bytes": experts + rows * (K * 16 + row + 2 * K * row + row), "flops": flops + 2.0 * rows * K * D}
    routed = 2 * E * D + experts
    flops += 2.0 * rows * E * D
    if kind == "verify":
        return {"bytes": routed + rows * (3 * row + 6 * K), "flops": flops}
    shared = 3 * _matrix_bytes(SHARED_F, D, case["shared_bits"])
    # rows: the tokens' table rows, attention's rows in, the residual stream out, the routes out; for a prompt, whose calls
    # return them, h1 and h2 as well
    per_row = _matrix_bytes(1, D) + 2 * row + 6 * K + (2 * row if kind == "prompt" else 0)
    return {"bytes": routed + shared + rows * per_row, "flops": flops + 2.0 * rows * 3 * D * SHARED_F}


def tolerance(case):
    # 16-bit results carry one rounding of the result and one of the activations between the two products
    if case["kind"] in ("greedy", "sample", "hot"):
        # fp32 sums over 2,816 products; a softmax probability is the exponential of such a sum
        return {"rel": 1e-4}
    return {"rel": 1e-2}
