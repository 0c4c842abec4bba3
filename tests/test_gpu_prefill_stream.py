"""The prefill's streaming product (chunks whose experts hold few pairs): experts with 0, 1 and every count around a 16-pair
block, around a tile of 32 and of 64 pairs, K of whole and of ragged chunks, output columns that do not fill an N-block, both
activation types, and the line between it and the grouped GEMMs. Needs a GPU: pytest -m gpu."""
import numpy as np
import pytest

from helpers import bf16_tensor, bits_of, cosine, make_layer, rel_err, to_ff_offsets

pytestmark = pytest.mark.gpu

COUNTS = (0, 1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 97, 130)


def _routes(rng, counts, e):
    """One route per token (top_k = 1), counts[i] tokens for expert i, tokens shuffled."""
    idx = np.repeat(np.arange(e, dtype=np.uint32), counts)
    rng.shuffle(idx)
    return idx[:, None]


# d, f: (groups of d, groups of f) = whole pairs of chunks, one ragged chunk, three groups past a pair; 320 columns = 2.5 N-blocks
@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("d,f,scale", [(256, 128, 1), (320, 192, 1), (448, 64, 2), (64, 704, 2), (320, 704, 1.5), (192, 576, 9)])
def test_tile_edges_against_the_oracle(oracle, act, d, f, scale):
    import torch
    import fieldfare_moe as ff
    ff.lib()
    # scale 1: 44 pairs per expert on average, 2: 22 (tiles of 32); 1.5: 29.5 and eleven N-blocks, more blocks than compute
    # units (tiles of 64); 9: 4.9 pairs and nine N-blocks, a tile of each expert between four and six blocks per unit (bf16: tiles of 16)
    e = int(len(COUNTS) * scale)
    counts = np.array(COUNTS + (0,) * (e - len(COUNTS)))
    rng, pool, _ = make_layer(oracle, 77 + d, d, f, e, align=1)
    idx = _routes(rng, counts, e)
    t = idx.shape[0]
    assert t <= 48 * e
    ctx = ff.Context(d, f, e, 1, n_layers=1, max_tokens=t, act_dtype=act)
    try:
        ctx.upload_layer(0, pool.bytes, pool.stride, to_ff_offsets(ff, pool.offsets))
        dt = torch.bfloat16 if act == "bf16" else torch.float16
        x = torch.from_numpy(rng.normal(0, 1, (t, d)).astype(np.float32)).to(dt)
        w = torch.from_numpy(rng.uniform(0.2, 1.0, (t, 1)).astype(np.float32)).to(dt)
        gi = torch.from_numpy(idx.view(np.int32)).cuda()
        y = ctx.prefill(0, x.cuda(), gi, w.cuda()).float().cpu().numpy()
        n_pairs, n_tiles, got_counts = ctx.prefill_stats()
        assert n_pairs == t and np.array_equal(got_counts, counts)
        assert n_tiles == int(np.sum((counts + ff.PREFILL_TILE_M - 1) // ff.PREFILL_TILE_M))       # the routes', not the chunk's own
        xf, wf = x.float().numpy(), w.float().numpy()
        ref, spread = np.zeros((t, d), np.float64), np.zeros((t, d), np.float64)
        for ex in range(e):
            rows = np.flatnonzero(idx[:, 0] == ex)
            if len(rows):
                g, u, dn = (oracle.dequantize_int4(*pool.sub(ex, n)).astype(np.float64) for n in ("gate", "up", "down"))
                gate, up = xf[rows] @ g.T, xf[rows] @ u.T
                act_rows = 0.5 * gate * (1 + np.tanh(0.7978845608028654 * (gate + 0.044715 * gate ** 3))) * up
                ref[rows] = wf[rows] * (act_rows @ dn.T)
                spread[rows] = wf[rows] * (np.abs(act_rows) @ np.abs(dn.T))
        # element by element: every activation rounded once (unit 2^-8 in bf16, 2^-11 in FP16, through the down product's
        # absolute sum), the per-route row and the weighted row once each; a tenth on top for the fp32 sums in the offset form
        unit = 2.0 ** (-8 if act == "bf16" else -11)
        assert np.all(np.abs(y - ref) <= 1.1 * unit * (spread + 2 * np.abs(ref)) + 1e-6 * np.abs(ref).max())
        # a pair's row does not depend on the pairs beside it: the chunk's first half alone, in tiles cut elsewhere
        half = t // 2
        part = ctx.prefill(0, x[:half].cuda(), gi[:half].contiguous(), w[:half].cuda()).float().cpu().numpy()
        assert np.array_equal(part, y[:half])
    finally:
        ctx.close()


# K of one to five chunks of two groups, the last one whole or ragged: every place at which the ring of row buffers can end, with four buffers
# (tiles of up to 32 pairs) and with three (tiles of 64)
@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("groups,f,scale", [(g, 128, 1) for g in (2, 6, 8, 9, 10)] + [(g, 704, 1.5) for g in (1, 2, 3, 4, 6, 7, 8)])
def test_the_ring_of_row_buffers_ends_anywhere(oracle, act, groups, f, scale):
    test_tile_edges_against_the_oracle(oracle, act, 64 * groups, f, scale)


def _exact_part(oracle, rows, cols, one_hot):
    """4-bit weights, scale 1 and bias 0, with q = 1 at column one_hot[row] and 0 elsewhere."""
    q = np.zeros((rows, cols), np.uint8)
    q[np.arange(rows), one_hot] = 1
    unit = oracle.bf16_bits(np.ones((rows, cols // 64), np.float32))
    return (q[:, ::2] | q[:, 1::2] << 4), unit, np.zeros_like(unit)


# one, two and (wide layers, tiles of 64 pairs) up to four 16-pair blocks per tile
@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("d,f,counts", [(256, 64, (9, 20, 32, 33)), (320, 128, (16, 17, 28, 1)), (1024, 704, 3 * (9, 20, 33, 40, 48, 49, 60, 16))])
@pytest.mark.parametrize("small", [0, 1, 3])
def test_a_small_group_beside_large_ones(oracle, act, d, f, counts, small):
    """One group of the up projection adds an odd whole number v, every other one nothing: q = 0 and bias 0 under scales of 2^7 and
    inputs of 8. There a bf16 sum is v + 2^23 for a moment (128 * 2^7 * 512), whole numbers that fp32 holds - not so v + 2^24,
    which two such groups at once would make. gate = 16 = gelu(16), down picks one activation per column: the rows are 16 v exactly."""
    import torch
    import fieldfare_moe as ff
    ff.lib()
    e, t, rng = len(counts), sum(counts), np.random.default_rng(d + small)
    assert 0 < t <= 48 * e
    cols = 64 * small + np.arange(1, 17)
    parts, v_of = [], []
    for _ in range(e):
        gate = _exact_part(oracle, f, d, np.full(f, 64 * small))
        gate[1][:] = oracle.bf16_bits(np.float32([16.0]))[0]
        q = np.zeros((f, d), np.uint8)
        q[:, cols] = rng.integers(0, 16, (f, 16))
        q[:, 64 * small] = 1 - q[:, cols].sum(1) % 2 + 14 * (rng.random(f) < 0.5)                       # makes the sum odd
        scale = np.full((f, d // 64), 128.0, np.float32)
        scale[:, small] = 1.0
        up = (q[:, ::2] | q[:, 1::2] << 4), oracle.bf16_bits(scale), np.zeros((f, d // 64), np.uint16)
        parts.append((gate, up, _exact_part(oracle, d, f, np.arange(d) % f)))
        v_of.append(q[:, 64 * small:64 * small + 17].astype(np.int64))
    idx = _routes(rng, counts, e)
    x = np.full((t, d), 8.0, np.float32)
    x[:, 64 * small:64 * small + 64] = 0
    x[:, 64 * small] = 1                                    # column 0 of the group: every row's
    pick = 2 * rng.integers(0, 2, (t, 16))                  # the others: 0 or 2, so that v stays odd where q of column 0 is
    x[:, cols] = pick
    ctx = ff.Context(d, f, e, 1, n_layers=1, max_tokens=t, act_dtype=act)
    try:
        pool = oracle.pool_from_parts(parts, d, f, 1, None)
        ctx.upload_layer(0, pool.bytes, pool.stride, to_ff_offsets(ff, pool.offsets))
        dt = torch.bfloat16 if act == "bf16" else torch.float16
        y = ctx.prefill(0, torch.from_numpy(x).to(dt).cuda(), torch.from_numpy(idx.view(np.int32)).cuda(), torch.ones((t, 1), dtype=dt).cuda())
        row_x = np.concatenate([np.ones((t, 1), np.int64), pick], 1)
        v = np.einsum("tk,tfk->tf", row_x, np.stack([v_of[i] for i in idx[:, 0]]))
        # (a whole number of more than 8 significant bits is rounded once, as the activation)
        want = torch.from_numpy(16.0 * v).to(torch.float32).to(dt).double().numpy()[:, np.arange(d) % f]
        assert np.array_equal(y.double().cpu().numpy(), want)
    finally:
        ctx.close()


# 1 to 5 groups of K in each product: a quad of groups short of three, two, one and none, and one group past it
@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("d,f", [(64, 128), (192, 64), (256, 192), (320, 256), (128, 320)])
def test_a_row_without_bounds_stays_alone(oracle, act, d, f):
    # an infinity or a NaN in a row (also in the last group, the one that loads past the end repeat): the others keep their bits
    import torch
    import fieldfare_moe as ff
    ff.lib()
    rng, pool, _ = make_layer(oracle, 3 * d + f, d, f, 4, align=1)
    dt = torch.bfloat16 if act == "bf16" else torch.float16
    t = 20
    x = torch.from_numpy(rng.normal(0, 1, (t, d)).astype(np.float32)).to(dt)
    idx = torch.from_numpy(np.stack([rng.permutation(4) for _ in range(t)]).astype(np.int32)).cuda()
    w = torch.full((t, 4), 0.25).to(dt).cuda()
    bad = x.clone()
    bad[3, d - 1], bad[17, 0] = float("inf"), float("nan")
    ctx = ff.Context(d, f, 4, 4, n_layers=1, max_tokens=t, act_dtype=act)
    try:
        ctx.upload_layer(0, pool.bytes, pool.stride, to_ff_offsets(ff, pool.offsets))
        y = ctx.prefill(0, x.cuda(), idx, w).cpu()
        z = ctx.prefill(0, bad.cuda(), idx, w).cpu()
        rest = [r for r in range(t) if r not in (3, 17)]
        assert torch.isfinite(y.float()).all() and torch.equal(y[rest].view(torch.int16), z[rest].view(torch.int16))
        assert not torch.isfinite(z[[3, 17]].float()).any()
    finally:
        ctx.close()


@pytest.mark.parametrize("t", [47, 48, 49])
def test_the_line_to_the_grouped_gemms(oracle, t):
    # four experts, top-4: t pairs each; 48 per expert is the last chunk that streams. Either side to the same bar.
    import torch
    import fieldfare_moe as ff
    ff.lib()
    d, f, e = 128, 128, 4
    rng, pool, _ = make_layer(oracle, 5, d, f, e, align=1)
    ctx = ff.Context(d, f, e, 4, n_layers=1, max_tokens=64)
    try:
        ctx.upload_layer(0, pool.bytes, pool.stride, to_ff_offsets(ff, pool.offsets))
        xb = oracle.bf16_bits(rng.normal(0, 1, (t, d)).astype(np.float32))
        idx = np.stack([rng.permutation(4) for _ in range(t)]).astype(np.uint32)
        wb = oracle.bf16_bits(rng.dirichlet(np.ones(4), size=t).astype(np.float32))
        y = oracle.bf16_to_float(bits_of(ctx.prefill(0, bf16_tensor(torch, xb), torch.from_numpy(idx.view(np.int32)).cuda(), bf16_tensor(torch, wb))))
        ref = oracle.moe_experts(pool, xb, idx, oracle.bf16_to_float(wb))
        assert rel_err(y, ref) <= 1e-2 and cosine(y, ref) >= 0.9999
    finally:
        ctx.close()


# 2,944 -> 2,816 (wider than the GEMV's ring, so from 17 rows on): one round of gate/up blocks up to 672 rows, bf16's products
# up to 796
@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("d,f,t", [(192, 320, 385), (192, 320, 895), (192, 320, 896), (192, 320, 897), (2944, 2816, 673), (2944, 2816, 797)])
def test_dense_chunks_beyond_the_gemv(oracle, act, d, f, t):
    # a dense FFN's chunk: tiles of 32 rows up to 896 rows, fewer where wide, the GEMMs from there on
    import torch
    import fieldfare_moe as ff
    ff.lib()
    g = oracle.seed_tree_key(0x5EED, f"dense-tiles-{t}")
    parts = tuple(oracle.quantize_int4(g.uniform(-0.3, 0.3, r * c).reshape(r, c)) for r, c in ((f, d), (f, d), (d, f)))
    x = torch.from_numpy(g.uniform(-1.0, 1.0, t * d).reshape(t, d).astype(np.float32)).to(torch.bfloat16 if act == "bf16" else torch.float16)
    ctx = ff.Context(d, f, 1, 1, n_layers=1, max_tokens=t, act_dtype=act)
    try:
        ctx.upload_expert_parts(0, 0, *parts)
        y = ctx.dense_ffn(0, x.cuda()).float().cpu().numpy()
        gw, uw, dw = (oracle.dequantize_int4(*p).astype(np.float64) for p in parts)
        xf = x.float().numpy()
        gate, up = xf @ gw.T, xf @ uw.T
        ref = (0.5 * gate * (1 + np.tanh(0.7978845608028654 * (gate + 0.044715 * gate ** 3))) * up) @ dw.T
        assert rel_err(y, ref) <= 1e-2 and cosine(y, ref) >= 0.9999
    finally:
        ctx.close()
