"""The prefill's grouped GEMMs: M-tiles of every number of 16-pair blocks (and one, two and no pairs past a block), plans whose
largest tile is at most half a tile, K of one group, of fewer and of more than the rings hold,
N-blocks that are full, half full and a quarter full, fewer and more items than compute units, both activation types; rows that
span more than 4 GiB. Needs a GPU: pytest -m gpu."""
import numpy as np
import pytest

from helpers import make_layer, to_ff_offsets

pytestmark = pytest.mark.gpu

LONG = (1, 16, 33, 64, 80, 96, 112, 113, 128, 129, 144, 160, 176, 177, 192, 208, 224, 240, 241, 255, 256, 257, 0, 300)
SHORT = (1, 15, 17, 32, 33, 64, 65, 80, 96, 97, 112, 113, 127, 128, 128, 0)


def _check(oracle, pool, e, idx, x, w, y, act):
    """Element by element against 64-bit products of the 16-bit tile weights: every activation rounded once (unit 2^-8 in bf16,
    2^-11 in FP16, through the down product's absolute sum), the per-route row and the weighted row once each; a tenth on top
    for the fp32 sums."""
    t, d = x.shape
    dt = x.dtype
    import torch
    unit = 2.0 ** (-8 if act == "bf16" else -11)
    xf, wf = x.double().numpy(), w.double().numpy()
    ref, spread = np.zeros((t, d)), np.zeros((t, d))
    for ex in range(e):
        rows = np.flatnonzero(idx[:, 0] == ex)
        if not len(rows):
            continue
        g, u, dn = (torch.from_numpy(oracle.dequantize_int4(*pool.sub(ex, n))).to(dt).double().numpy() for n in ("gate", "up", "down"))
        gate, up = xf[rows] @ g.T, xf[rows] @ u.T
        act_rows = 0.5 * gate * (1 + np.tanh(0.7978845608028654 * (gate + 0.044715 * gate ** 3))) * up
        ref[rows] = wf[rows] * (act_rows @ dn.T)
        spread[rows] = wf[rows] * (np.abs(act_rows) @ np.abs(dn.T))
    assert np.all(np.abs(y - ref) <= 1.1 * unit * (spread + 2 * np.abs(ref)) + 1e-6 * np.abs(ref).max())


@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("d,f,counts", [(64, 2816, LONG), (128, 1408, LONG), (192, 320, LONG), (704, 192, LONG), (2816, 64, LONG),
                                        (1408, 128, LONG), (320, 704, LONG), (704, 320, SHORT), (2816, 128, SHORT), (192, 2816, SHORT)])
def test_tiles_and_rings_against_the_oracle(oracle, act, d, f, counts):
    import torch
    import fieldfare_moe as ff
    ff.lib()
    e = len(counts)
    rng, pool, _ = make_layer(oracle, 31 + d + f, d, f, e, align=1)
    idx = np.repeat(np.arange(e, dtype=np.uint32), counts)
    rng.shuffle(idx)
    idx = idx[:, None]
    t = idx.shape[0]
    assert t > 48 * e
    ctx = ff.Context(d, f, e, 1, n_layers=1, max_tokens=t, act_dtype=act)
    try:
        ctx.upload_layer(0, pool.bytes, pool.stride, to_ff_offsets(ff, pool.offsets))
        dt = torch.bfloat16 if act == "bf16" else torch.float16
        x = torch.from_numpy(rng.normal(0, 1, (t, d)).astype(np.float32)).to(dt)
        w = torch.from_numpy(rng.uniform(0.2, 1.0, (t, 1)).astype(np.float32)).to(dt)
        gi = torch.from_numpy(idx.view(np.int32)).cuda()
        y = ctx.prefill(0, x.cuda(), gi, w.cuda())
        _check(oracle, pool, e, idx, x, w, y.float().cpu().numpy(), act)
        # the chunk backwards: other pairs in every tile, the same rows
        back = ctx.prefill(0, x.flip(0).cuda(), gi.flip(0).contiguous(), w.flip(0).cuda())
        assert torch.equal(back.flip(0), y)
    finally:
        ctx.close()


# Tiles of fewer than 256 pairs, where few experts leave compute units idle: of 128, 64 and 32 pairs, all of a chunk in one expert (as
# many tiles as there can be), one expert, no more than a uniform chunk's experts have (80); and whole tiles on long gate/up rings, which take more items than there are units.
@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("d,f,counts", [(320, 1536, (192, 130, 256, 257, 128, 1, 0, 300)), (320, 1536, (0, 0, 1300, 0, 0, 3, 0, 0)),
                                        (320, 1536, (63, 64, 65, 31, 96, 129, 0, 128)), (192, 320, (1000, 24)), (192, 320, (31, 32, 33, 65, 96, 97)),
                                        (448, 384, (700,)), (448, 384, (290,)), (192, 1536, (700,) + 15 * (9,)), (192, 1536, (1900,) + 39 * (5,)), (192, 704, LONG), (1408, 704, LONG)])
def test_tiles_by_the_number_of_items(oracle, act, d, f, counts):
    test_tiles_and_rings_against_the_oracle(oracle, act, d, f, counts)


# Chunks of more than one round in tiles of 96 and 112 pairs, two blocks per compute unit: the edges of 16-pair blocks, experts that such a
# tile does not hold, tall and flat layers, a last N-block that is half full. The same rows three times over take larger tiles: the same bits.
@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("d,f,counts", [(192, 704, 8 * (1, 16, 47, 64, 127, 128, 129, 0)), (64, 640, 8 * (17, 33, 80, 81, 96, 112, 113, 0)),
                                        (512, 704, 7 * (31, 65, 48, 97, 95, 100, 63) + (257, 15))])
def test_tiles_of_half_the_pairs(oracle, act, d, f, counts):
    import torch
    import fieldfare_moe as ff
    ff.lib()
    e, t = len(counts), sum(counts)
    assert 48 * e < t <= 112 * e and 3 * t > 130 * e
    rng, pool, _ = make_layer(oracle, 51 + d, d, f, e, align=1)
    idx = np.repeat(np.arange(e, dtype=np.uint32), counts)
    rng.shuffle(idx)
    ctx = ff.Context(d, f, e, 1, n_layers=1, max_tokens=3 * t, act_dtype=act)
    try:
        ctx.upload_layer(0, pool.bytes, pool.stride, to_ff_offsets(ff, pool.offsets))
        dt = torch.bfloat16 if act == "bf16" else torch.float16
        x = torch.from_numpy(rng.normal(0, 1, (t, d)).astype(np.float32)).to(dt)
        w = torch.from_numpy(rng.uniform(0.2, 1.0, (t, 1)).astype(np.float32)).to(dt)
        gx, gi, gw = x.cuda(), torch.from_numpy(idx[:, None].view(np.int32)).cuda(), w.cuda()
        tall = ctx.prefill(0, gx.repeat(3, 1), gi.repeat(3, 1), gw.repeat(3, 1))
        ctx.prefill(0, torch.full_like(gx, float("nan")), gi, gw)           # (nothing of the rows stays in the scratch)
        y = ctx.prefill(0, gx, gi, gw, out=torch.full_like(gx, float("nan")))
        _check(oracle, pool, e, idx[:, None], x, w, y.float().cpu().numpy(), act)
        assert all(torch.equal(tall[k * t:(k + 1) * t], y) for k in range(3))
    finally:
        ctx.close()


# Layers of more than two rounds of items (576 or 640 gate/up N-blocks for 256 units), where a chunk of up to some 112 pairs per expert is cut
# at 128: one pair around a 16-pair block, around one tile and two; every expert one pair past a tile, as many tiles as there can be.
@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("d,f,counts", [(128, 704, 12 * (112, 113, 127, 128, 129, 96, 60, 81)), (64, 640, 16 * (257, 112, 113, 128, 127, 129, 1, 17)),
                                        (64, 704, 48 * (129, 81))])
def test_tiles_of_128_pairs_where_the_chip_is_full(oracle, act, d, f, counts):
    e, t = len(counts), sum(counts)
    assert e * ((f // 16 + 7) // 8) > 2 * 256 and 48 * e < t and t / e + 1.5 * (t / e) ** 0.5 <= 128
    test_tiles_and_rings_against_the_oracle(oracle, act, d, f, counts)


@pytest.mark.parametrize("act,stride", [("bf16", 1 << 24), ("bf16", 1 << 25), ("fp16", 1 << 25), ("bf16", 360_000_000), ("fp16", 360_000_000)])
def test_rows_that_span_four_gigabytes(oracle, act, stride):
    # 99 rows 32 MiB apart: a place past 2 GiB; 64 MiB: a row's place in bytes does not fit 32 bits; 720 MB apart: nor does the one in 16-byte pieces
    import torch
    import fieldfare_moe as ff
    ff.lib()
    d, f, e, t = 256, 192, 2, 99
    if torch.cuda.mem_get_info()[0] < t * stride * 2 + (4 << 30):
        pytest.skip("the card's free memory does not hold the rows")
    rng, pool, _ = make_layer(oracle, 9, d, f, e, align=1)
    ctx = ff.Context(d, f, e, 1, n_layers=1, max_tokens=t, act_dtype=act)
    try:
        ctx.upload_layer(0, pool.bytes, pool.stride, to_ff_offsets(ff, pool.offsets))
        dt = torch.bfloat16 if act == "bf16" else torch.float16
        x = torch.from_numpy(rng.normal(0, 1, (t, d)).astype(np.float32)).to(dt).cuda()
        idx = torch.from_numpy(rng.integers(0, e, (t, 1)).astype(np.int32)).cuda()
        w = torch.from_numpy(rng.uniform(0.2, 1.0, (t, 1)).astype(np.float32)).to(dt).cuda()
        far = torch.empty(((t - 1) * stride + d,), dtype=dt, device="cuda").as_strided((t, d), (stride, 1))
        far.copy_(x)
        near = ctx.prefill(0, x, idx, w)
        assert torch.isfinite(near).all() and near.abs().max() > 0
        ctx.prefill(0, -x, idx, w)                              # (nothing of the rows stays in the scratch)
        assert torch.equal(ctx.prefill(0, far, idx, w, out=torch.full_like(near, float("nan"))), near)
    finally:
        ctx.close()
        far = None
        torch.cuda.empty_cache()


# Rows 8 and 4 MiB apart, 5 to 7.4 GB in all, of nine experts with 288 gate/up N-blocks: about 67 pairs per expert in tiles of 112, about 98 in
# tiles of 128 (with 113, 127, 128 and more), about 150 in tiles of 208.
@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("counts,stride", [((112, 97, 80, 64, 48, 33, 100, 40, 26), 1 << 22), ((128, 113, 127, 112, 129, 80, 97, 64, 33), 1 << 22),
                                           ((208, 193, 177, 145, 129, 209, 113, 96, 80), 1 << 21)])
def test_far_rows_in_tiles_of_every_height(oracle, act, counts, stride):
    import torch
    import fieldfare_moe as ff
    ff.lib()
    d, f, e, t = 128, 4096, len(counts), sum(counts)
    assert t * stride * 2 > 1 << 32 and t > 48 * e and e * f // 128 > 256
    if torch.cuda.mem_get_info()[0] < t * stride * 2 + (4 << 30):
        pytest.skip("the card's free memory does not hold the rows")
    rng, pool, _ = make_layer(oracle, 13, d, f, e, align=1)
    idx = np.repeat(np.arange(e, dtype=np.uint32), counts)
    rng.shuffle(idx)
    ctx = ff.Context(d, f, e, 1, n_layers=1, max_tokens=t, act_dtype=act)
    try:
        ctx.upload_layer(0, pool.bytes, pool.stride, to_ff_offsets(ff, pool.offsets))
        dt = torch.bfloat16 if act == "bf16" else torch.float16
        x = torch.from_numpy(rng.normal(0, 1, (t, d)).astype(np.float32)).to(dt)
        w = torch.from_numpy(rng.uniform(0.2, 1.0, (t, 1)).astype(np.float32)).to(dt)
        gx, gi, gw = x.cuda(), torch.from_numpy(idx[:, None].view(np.int32)).cuda(), w.cuda()
        far = torch.empty(((t - 1) * stride + d,), dtype=dt, device="cuda").as_strided((t, d), (stride, 1))
        far.copy_(gx)
        near = ctx.prefill(0, gx, gi, gw)
        _check(oracle, pool, e, idx[:, None], x, w, near.float().cpu().numpy(), act)
        ctx.prefill(0, -gx, gi, gw)                             # (nothing of the rows stays in the scratch)
        assert torch.equal(ctx.prefill(0, far, gi, gw, out=torch.full_like(near, float("nan"))), near)
    finally:
        ctx.close()
        far = None
        torch.cuda.empty_cache()


@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("d,f,rows", [(704, 1408, (897, 1025, 1500, 1601, 2049, 2300, 2800, 3000, 3600, 4000, 4400, 5000)),
                                      (1408, 1408, (913, 1700, 4801, 5000, 5600)), (2816, 704, (1200, 2048, 3000, 4096))])
def test_dense_tiles_of_the_row_count(oracle, act, d, f, rows):
    """A dense FFN's tiles have as many rows as fill the last round of blocks (64 to 256; over 2,560 columns and more, tiles of 96 and 112 rows run
    a block per compute unit): the largest chunk against 64-bit products, every other one, cut elsewhere, to the same bits."""
    import torch
    import fieldfare_moe as ff
    ff.lib()
    rng, pool, _ = make_layer(oracle, 77 + d, d, f, 1, align=1)
    t = max(rows)
    ctx = ff.Context(d, f, 1, 1, n_layers=1, max_tokens=t, act_dtype=act)
    try:
        ctx.upload_layer(0, pool.bytes, pool.stride, to_ff_offsets(ff, pool.offsets))
        dt = torch.bfloat16 if act == "bf16" else torch.float16
        x = torch.from_numpy(rng.normal(0, 1, (t, d)).astype(np.float32)).to(dt)
        y = ctx.dense_ffn(0, x.cuda())
        # (the reference's cost bounds the rows compared: the first and last of the chunk, which every tile size cuts differently)
        some = np.r_[0:200, t - 200:t]
        _check(oracle, pool, 1, np.zeros((len(some), 1), np.uint32), x[some], torch.ones((len(some), 1), dtype=dt), y.float().cpu().numpy()[some], act)
        for n in rows:
            # (after rows of NaN through the scratch and into NaN: what is not written is not equal)
            ctx.dense_ffn(0, torch.full_like(x, float("nan")).cuda())
            assert torch.equal(ctx.dense_ffn(0, x[:n].cuda(), out=torch.full_like(y[:n], float("nan"))), y[:n]), n
    finally:
        ctx.close()
