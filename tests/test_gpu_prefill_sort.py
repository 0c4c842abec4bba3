"""The prefill's sort of routes in one launch (up to 16,384 to 65,536 items) and in three: the same rows, bit for bit, from a chunk and from its
beginning, on one side of the line and on either, and from lists of pairs, counts per expert, routes of weight zero and experts past the last left
out (on either side of the line). What a call does not write is NaN. (The order of an expert's pairs shows in no result.) Needs a GPU: pytest -m gpu."""
import numpy as np
import pytest

from helpers import make_layer, to_ff_offsets

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("e,k,cuts", [(128, 8, (1, 7, 8, 9, 128, 129, 383, 384)), (256, 2, (31, 32, 33, 511, 512, 513, 1535, 1536)),
                                      (3, 1, (3000, 3071, 3072)), (5, 3, (1024,)), (200, 4, (255, 256, 257, 768))])
def test_chunks_and_their_beginnings(oracle, e, k, cuts):
    import torch
    import fieldfare_moe as ff
    ff.lib()
    d, f, t = 128, 64, 3072 // k + 5
    rng, pool, _ = make_layer(oracle, 3 + e, d, f, e, align=1)
    idx = np.stack([rng.permutation(e)[:k] for _ in range(t)]).astype(np.uint32)
    w = rng.uniform(0.2, 1.0, (t, k)).astype(np.float32)
    w[rng.random((t, k)) < 0.05] = 0
    ctx = ff.Context(d, f, e, k, n_layers=1, max_tokens=t)
    try:
        ctx.upload_layer(0, pool.bytes, pool.stride, to_ff_offsets(ff, pool.offsets))
        x = torch.from_numpy(rng.normal(0, 1, (t, d)).astype(np.float32)).to(torch.bfloat16).cuda()
        gi, gw = torch.from_numpy(idx.view(np.int32)).cuda(), torch.from_numpy(w).to(torch.bfloat16).cuda()
        def counts(n, routes):
            live = (w[:n] > 0) & (routes[:n] < e)
            return np.bincount(routes[:n][live], minlength=e)

        def rows(n, routes, weights):
            # whatever a lost or doubled route leaves unwritten is NaN: the routes' rows in the scratch and the output rows
            ctx.prefill(0, torch.full_like(x, float("nan")), gi, torch.ones_like(gw))
            y = ctx.prefill(0, x[:n], routes[:n].contiguous(), weights[:n].contiguous(), out=torch.full_like(x[:n], float("nan")))
            return y, ctx.prefill_stats()

        whole, stats = rows(t, gi, gw)                          # 3,072 + 5 k items
        assert torch.isfinite(whole.float()).all() and whole.abs().max() > 0
        assert np.array_equal(stats[2], counts(t, idx))
        for n in cuts:                                          # (the same products as the whole chunk's: equal bit for bit)
            part, stats = rows(n, gi, gw)
            assert np.array_equal(stats[2], counts(n, idx)), n
            assert torch.equal(part, whole[:n]), n
        # experts past the last: as if the routes had weight zero
        lost = rng.random((t, k)) < 0.2
        past = torch.from_numpy(np.where(lost, e + 3, idx).astype(np.int32)).cuda()
        less = gw.masked_fill(torch.from_numpy(lost).cuda(), 0)
        for n in (cuts[-1], t):
            got, (n_pairs, _, per_expert) = rows(n, past, gw)
            assert np.array_equal(per_expert, counts(n, np.where(lost, e + 3, idx))) and n_pairs == per_expert.sum(), n
            assert torch.equal(got, rows(n, gi, less)[0]), n
        # a list of pairs in any order, its first 3,072 and all of it: the rows that are listed, no others
        token, rank = (v.reshape(-1) for v in np.divmod(rng.permutation(t * k), k))
        lists = np.stack([token, np.where((w > 0) & ~lost, idx, e + 3)[token, rank], rank, np.zeros_like(token)], 1).astype(np.int32)
        kept = torch.from_numpy(lists[:, 1] < e).cuda()
        got = []
        for n in (t * k, 3072):
            ctx.prefill(0, torch.full_like(x, float("nan")), gi, torch.ones_like(gw))
            out = torch.full((t * k, d), float("nan"), dtype=x.dtype, device="cuda")
            ctx.prefill_pairs(0, x, torch.from_numpy(lists[:n].copy()).cuda(), t, out)
            assert np.array_equal(ctx.prefill_stats()[2], np.bincount(lists[:n, 1], minlength=e + 4)[:e]), n
            got.append(out[torch.from_numpy(token * k + rank).cuda()])      # in the list's order
        all_rows, first = got
        assert torch.isfinite(all_rows[kept]).all() and torch.isnan(all_rows[~kept]).all()
        assert torch.equal(first[:3072][kept[:3072]], all_rows[:3072][kept[:3072]])
        assert torch.isnan(first[3072:]).all() and torch.isnan(first[:3072][~kept[:3072]]).all()
    finally:
        ctx.close()


@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("t,k,d,skip", [(1, 1, 8, 0), (3, 8, 2816, 0), (33, 8, 72, 0), (5, 9, 64, 0), (7, 17, 1000, 0), (5, 3, 13, 0), (9, 8, 64, 1), (300, 2, 8, 0)])
def test_reduce_of_rows_by_pieces_and_by_elements(oracle, act, t, k, d, skip):
    # 16-byte pieces where width and addresses allow, elements elsewhere: the oracle's fma in rank order, bit for bit
    import torch
    import fieldfare_moe as ff
    ff.lib()
    dt, kind = (torch.bfloat16, oracle.BF16) if act == "bf16" else (torch.float16, oracle.FP16)
    rng = np.random.default_rng(t * 100 + k)
    ctx = ff.Context(64, 64, 4, 1, n_layers=1, max_tokens=16, act_dtype=act)
    try:
        flat = torch.from_numpy(rng.normal(0, 1, t * k * d + skip).astype(np.float32)).to(dt).cuda()
        partials = flat[skip:].view(t, k, d)
        w = torch.from_numpy(rng.normal(0, 1, (t, k)).astype(np.float32)).to(dt).cuda()
        bits = lambda a: a.view(torch.int16).cpu().numpy().view(np.uint16)
        got = bits(ctx.reduce_token_major(partials, w))
        assert np.array_equal(got, oracle.reduce_token_major(bits(partials), kind, bits(w), kind))
    finally:
        ctx.close()


# the last item count of one launch and the first of three (20,480 items with up to 64 experts, 24,576 with up to 128 and 65,536 beyond)
# and past it, runs of 64 items per wave that end inside a group of eight loads, and the few items that 256 threads sort (2,048)
@pytest.mark.parametrize("e,k,line,cuts", [(64, 4, 20480, (682, 683, 5120)), (65, 3, 24576, (8191, 8192)), (128, 1, 24576, (2047, 2049, 24576)), (24, 2, 20480, (1023, 1025, 4500, 10240)), (33, 3, 24576, (682, 683, 2731, 8192)), (250, 8, 65536, (255, 257, 4097, 8192))])
def test_one_launch_at_its_line(oracle, e, k, line, cuts):
    import torch
    import fieldfare_moe as ff
    ff.lib()
    d, f, t = 64, 64, line // k + 3
    rng, pool, _ = make_layer(oracle, 5 + e, d, f, e, align=1)
    idx = np.argsort(rng.random((t, e)) - np.linspace(0, 0.6, e) * (rng.random((t, 1)) < 0.5), axis=1)[:, :k].astype(np.uint32)     # uneven
    w = rng.uniform(0.2, 1.0, (t, k)).astype(np.float32)
    w[rng.random((t, k)) < 0.05] = 0
    ctx = ff.Context(d, f, e, k, n_layers=1, max_tokens=t)
    try:
        ctx.upload_layer(0, pool.bytes, pool.stride, to_ff_offsets(ff, pool.offsets))
        x = torch.from_numpy(rng.normal(0, 1, (t, d)).astype(np.float32)).to(torch.bfloat16).cuda()
        gi, gw = torch.from_numpy(idx.view(np.int32)).cuda(), torch.from_numpy(w).to(torch.bfloat16).cuda()

        def rows(n):
            # what a lost or doubled route leaves unwritten is NaN
            ctx.prefill(0, torch.full_like(x, float("nan")), gi, torch.ones_like(gw))
            y = ctx.prefill(0, x[:n], gi[:n].contiguous(), gw[:n].contiguous(), out=torch.full_like(x[:n], float("nan")))
            n_pairs, n_tiles, counts = ctx.prefill_stats()
            assert np.array_equal(counts, np.bincount(idx[:n][w[:n] > 0], minlength=e)) and n_pairs == counts.sum(), n
            assert n_tiles == int(np.sum((counts + ff.PREFILL_TILE_M - 1) // ff.PREFILL_TILE_M)), n
            return y

        whole = rows(t)                                         # three launches
        assert torch.isfinite(whole.float()).all() and whole.abs().max() > 0
        assert torch.equal(rows(line // k), whole[:line // k])  # one launch where the line is this table's, the same products
        for n in cuts:                                          # (in the streaming product's range to its own bits: rounded weights elsewhere)
            part = rows(n)
            close = (part.float() - whole[:n].float()).abs() <= 2.0 ** -6 * whole[:n].float().abs() + 2.0 ** -6 * whole.float().abs().max()
            assert close.all(), n
    finally:
        ctx.close()


# (lists: one launch up to 20,480 pairs with up to four experts, 16,384 with up to 128, 65,536 beyond)
@pytest.mark.parametrize("e,k,line", [(4, 2, 20480), (5, 2, 16384), (128, 3, 16384), (24, 2, 20480), (33, 3, 24576), (250, 8, 65536)])
def test_lists_and_lost_routes_past_the_line(oracle, e, k, line):
    """What the three launches leave out and what they take: a list in any order, the same in order, its first part in one launch; a table
    with experts past the last against the same with weight zero."""
    import torch
    import fieldfare_moe as ff
    ff.lib()
    d, f, t = 64, 64, line // k + 3
    rng, pool, _ = make_layer(oracle, 15 + e, d, f, e, align=1)
    idx = np.argsort(rng.random((t, e)), axis=1)[:, :k].astype(np.int64)
    token, rank = (v.reshape(-1) for v in np.divmod(rng.permutation(t * k), k))
    lists = np.stack([token, idx[token, rank], rank, np.zeros_like(token)], 1).astype(np.int32)
    lost = rng.random(t * k) < 0.05
    lists[np.flatnonzero(lost), rng.integers(0, 3, lost.sum())] += 1 << 20          # each a token, an expert or a rank past the last
    in_order = lists[np.argsort(lists[:, 1], kind="stable")]
    ctx = ff.Context(d, f, e, k, n_layers=1, max_tokens=t)
    try:
        ctx.upload_layer(0, pool.bytes, pool.stride, to_ff_offsets(ff, pool.offsets))
        x = torch.from_numpy(rng.normal(0, 1, (t, d)).astype(np.float32)).to(torch.bfloat16).cuda()

        def rows(pairs, kept):
            out = torch.full((t * k, d), float("nan"), dtype=x.dtype, device="cuda")
            ctx.prefill_pairs(0, x, torch.from_numpy(pairs.copy()).cuda(), t, out)
            n_pairs, _, counts = ctx.prefill_stats()
            assert n_pairs == kept.sum() and np.array_equal(counts, np.bincount(lists[:len(kept)][kept, 1], minlength=e))
            return out.view(torch.int16)

        assert t * k > line
        three, sorted_three, one = rows(lists, ~lost), rows(in_order, ~lost), rows(lists[:line], ~lost[:line])
        assert torch.equal(three, sorted_three)                 # NaN where nothing is written, on both
        place = torch.from_numpy(token * k + rank).cuda()
        written = torch.isfinite(three.view(x.dtype)[place]).all(1).cpu().numpy()
        assert np.array_equal(written, ~lost)
        assert torch.equal(one[place[:line]], three[place[:line]]) and torch.isnan(one.view(x.dtype)[place[line:]]).all()

        gone = rng.random((t, k)) < 0.2
        past = torch.from_numpy(np.where(gone, e + rng.integers(0, 1 << 20, (t, k)), idx).astype(np.int32)).cuda()
        plain, w = torch.from_numpy(idx.astype(np.int32)).cuda(), torch.from_numpy(rng.uniform(0.2, 1.0, (t, k)).astype(np.float32)).to(x.dtype)
        less, w = w.masked_fill(torch.from_numpy(gone), 0).cuda(), w.cuda()
        for n in (t, line // k):                                # three launches, one
            ctx.prefill(0, torch.full_like(x, float("nan")), plain, torch.ones_like(w))
            got = ctx.prefill(0, x[:n], past[:n].contiguous(), w[:n].contiguous(), out=torch.full_like(x[:n], float("nan")))
            n_pairs, _, counts = ctx.prefill_stats()
            assert n_pairs == (~gone[:n]).sum() and np.array_equal(counts, np.bincount(idx[:n][~gone[:n]], minlength=e)), n
            assert torch.isfinite(got.float()).all() and torch.equal(got, ctx.prefill(0, x[:n], plain[:n].contiguous(), less[:n].contiguous())), n
    finally:
        ctx.close()


# 256 threads (2,048 pairs and fewer) and 1,024, runs of 64 pairs that end in one expert, in several and in pairs that are left out
@pytest.mark.parametrize("e,k,n", [(128, 8, 8000), (128, 8, 2048), (3, 2, 2049), (200, 1, 130), (7, 4, 63), (1, 1, 700)])
def test_lists_sorted_by_expert(oracle, e, k, n):
    import torch
    import fieldfare_moe as ff
    ff.lib()
    d, f, t = 64, 64, (n + k - 1) // k + 40
    rng, pool, _ = make_layer(oracle, 9 + e, d, f, e, align=1)
    idx = np.stack([rng.permutation(e)[:k] for _ in range(t)])
    token, rank = (v.reshape(-1) for v in np.divmod(rng.permutation(t * k)[:n], k))
    lists = np.stack([token, idx[token, rank], rank, np.zeros_like(token)], 1).astype(np.int32)
    out_of_range = rng.random(n) < 0.05
    lists[np.flatnonzero(out_of_range), rng.integers(0, 3, out_of_range.sum())] += 1 << 20          # each a token, an expert or a rank past the last
    in_order = lists[np.argsort(lists[:, 1], kind="stable")]
    ctx = ff.Context(d, f, e, k, n_layers=1, max_tokens=t)
    try:
        ctx.upload_layer(0, pool.bytes, pool.stride, to_ff_offsets(ff, pool.offsets))
        x = torch.from_numpy(rng.normal(0, 1, (t, d)).astype(np.float32)).to(torch.bfloat16).cuda()
        got = []
        for pairs in (lists, in_order):
            out = torch.full((t * k, d), float("nan"), dtype=x.dtype, device="cuda")
            ctx.prefill_pairs(0, x, torch.from_numpy(pairs.copy()).cuda(), t, out)
            n_pairs, _, counts = ctx.prefill_stats()
            assert n_pairs == n - out_of_range.sum() and np.array_equal(counts, np.bincount(lists[~out_of_range, 1], minlength=e))
            got.append(out.view(torch.int16))
        assert torch.equal(got[0], got[1])                       # NaN where nothing is written, on both
        written = torch.isfinite(out).all(1).cpu().numpy()
        assert np.array_equal(np.flatnonzero(written), np.sort((token * k + rank)[~out_of_range]))
    finally:
        ctx.close()
