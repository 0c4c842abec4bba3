"""Dense FFNs of 17 rows to a few hundred in bands of input rows: a row has the bits of the 16-row pass (8 bits) and of the same row
in any other chunk (4 bits), in every split of K and number of row blocks per band, at K of one group and of no multiple of the
splits, tile counts that fill no block, both activation types. Needs a GPU: pytest -m gpu."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(64, 64, (17, 33, 191)), (320, 192, (31, 64, 190)), (576, 2816, (17, 40, 97, 129, 161, 191)), (2816, 576, (18, 47, 129, 191)),
          (2816, 2816, (17, 32, 33, 49, 65, 81, 97, 129, 145, 177, 191)), (192, 1472, (100, 191)), (64, 1536, (17, 32, 33)), (192, 1600, (17, 32, 33))]


def _context(ff, oracle, torch, act, d, f, bits, cap):
    g = oracle.seed_tree_key(0xBA2D, f"bands-{d}-{f}-{bits}")
    quantize = oracle.quantize_int8 if bits == 8 else oracle.quantize_int4
    parts = tuple(quantize(g.uniform(-0.1, 0.1, r * c).reshape(r, c)) for r, c in ((f, d), (f, d), (d, f)))
    x = torch.from_numpy(g.uniform(-1.0, 1.0, cap * d).reshape(cap, d).astype(np.float32)).to(torch.bfloat16 if act == "bf16" else torch.float16)
    ctx = ff.Context(d, f, 1, 1, n_layers=1, max_tokens=cap, act_dtype=act)
    ctx.upload_expert_parts(0, 0, *parts, int8=bits == 8)
    return ctx, x.cuda()


@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("d,f,rows", SHAPES)
def test_8_bit_rows_equal_the_16_row_pass(oracle, act, d, f, rows):
    import torch
    import fieldfare_moe as ff
    ff.lib()
    ctx, x = _context(ff, oracle, torch, act, d, f, 8, 191)
    try:
        want = torch.cat([ctx.dense_ffn(0, x[r:r + 16]).clone() for r in range(0, 191, 16)])
        assert torch.isfinite(want).all() and want.abs().max() > 0
        for t in rows:
            assert torch.equal(ctx.dense_ffn(0, x[:t]), want[:t]), t
            # rows that are apart, and the last ones
            wide = torch.full((t, 2 * d + 8), float("nan"), dtype=x.dtype, device="cuda")
            wide[:, :d] = x[191 - t:]
            assert torch.equal(ctx.dense_ffn(0, wide[:, :d]), want[191 - t:]), t
    finally:
        ctx.close()


@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("d,f,rows", [(d, f, rows + (250, 301, 383)) for d, f, rows in SHAPES])
def test_4_bit_rows_equal_other_chunks(oracle, act, d, f, rows):
    import torch
    import fieldfare_moe as ff
    ff.lib()
    ctx, x = _context(ff, oracle, torch, act, d, f, 4, 384)
    try:
        want = torch.cat([ctx.dense_ffn(0, x[r:r + 24]).clone() for r in range(0, 384, 24)])
        assert torch.isfinite(want).all() and want.abs().max() > 0
        for t in rows:
            assert torch.equal(ctx.dense_ffn(0, x[:t]), want[:t]), t
            assert torch.equal(ctx.dense_ffn(0, x[384 - t:]), want[384 - t:]), t
    finally:
        ctx.close()


# more rows than the line below which bands always serve: where they are the faster (narrow layers) a row keeps the bits that it has in
# chunks below the line; where the other form is (rows past the last of a shape's range) it comes within both forms' roundings of them
@pytest.mark.parametrize("d,f,bits,rows", [(1024, 512, 4, (385, 512, 896)), (2816, 704, 4, (385, 640)), (192, 320, 4, (400, 895, 897)), (2816, 2816, 4, (400, 560)),
                                           (1024, 512, 8, (192, 301, 511)), (192, 320, 8, (192, 639)), (2048, 1408, 8, (192, 448, 560)), (2816, 2112, 8, (192, 208, 240, 301, 384, 385))])
def test_rows_past_the_lines(oracle, d, f, bits, rows):
    import torch
    import fieldfare_moe as ff
    ff.lib()
    past = {(192, 320, 4): 896, (2816, 2816, 4): 512, (2816, 2112, 8): 240, (2048, 1408, 8): 512}.get((d, f, bits), max(rows))
    ctx, x = _context(ff, oracle, torch, "bf16", d, f, bits, max(rows))
    try:
        want = torch.cat([ctx.dense_ffn(0, x[r:r + 160]).clone() for r in range(0, max(rows), 160)])
        assert torch.isfinite(want).all() and want.abs().max() > 0
        for t in rows:
            got = ctx.dense_ffn(0, x[:t])
            if t <= past:
                assert torch.equal(got, want[:t]), t
            else:
                # one rounding of the weights or of each activation more on either side (2^-9 of a term), and the rows' own (2^-9): within
                # 2^-6 of the largest row
                assert (got.float() - want[:t].float()).abs().max() <= 2.0 ** -6 * want.float().abs().max(), t
    finally:
        ctx.close()
