"""The listed GEMV on the matrix unit at the edges of its blocks (16 weight rows), parts of K (eight of up to six groups) and forms (up to
four input rows or more, aligned weights and rows or not). Needs a GPU: pytest -m gpu."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("m,n,shift", [(1, 64, 0), (15, 448, 0), (16, 512, 2), (17, 576, 0), (33, 2752, 2), (8193, 2816, 0), (8209, 320, 2)])
def test_listed_forms_agree(m, n, shift, act):
    import torch
    import fieldfare_moe as ff
    from fieldfare_moe import synthetic as syn
    gen = torch.Generator(device="cuda")
    gen.manual_seed(m + n)
    ctx = ff.Context(128, 64, 16, 8, n_layers=1, max_tokens=16, act_dtype=act)
    table = m + 7
    W, S, B = syn.synth_matrix_gpu(torch, gen, table, n)
    if shift:       # weight rows that are aligned to two bytes only
        room = torch.empty(W.numel() + shift, dtype=torch.uint8, device="cuda")
        room[shift:] = W.flatten()
        W = room[shift:].view(W.shape)
    ids = torch.randint(0, table, (m,), device="cuda", generator=gen, dtype=torch.int32)
    pad = 1 if shift and act == "bf16" else 8       # (FP16 rows have to come aligned)
    x = torch.randn((16, n + pad), device="cuda", generator=gen).to(ctx.act)[:, :n]
    q = torch.stack((W & 15, W >> 4), 2).view(table, n).double()
    s, b = (t.double().repeat_interleave(64, 1) for t in (S, B))
    rows = ids.long()
    want = x.double() @ (q * s + b)[rows].T
    # A group's sum holds 64 products of x with 16 + q (bf16) or q (FP16) in fp32, then a scale and a bias per group and the eight parts: no
    # more roundings than that on any path, each of 2^-24 (one bit more where the matrix unit truncates) of no more than the sum of magnitudes.
    offset = 0 if act == "fp16" else 16
    size = x.double().abs() @ ((2 * offset + q) * s + b.abs())[rows].T
    bound = size * 2.0 ** -23 * (64 + 2 * (n // 64) + 7)
    of = {}
    for r in (16, 5, 4, 1):
        y = ctx.gemv_int4_listed(W, S, B, ids, x[:r])
        assert ((y.double() - want[:r]).abs() <= bound[:r]).all(), r
        of[r] = y
        assert torch.equal(y, of[16][:r]), r       # whatever the form, a row's bits are the same
    ctx.close()


@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("rows", [1, 4, 5, 16])
def test_a_block_for_every_sixteen_rows_or_not(act, rows):
    # up to 32 weight rows per compute unit a block takes sixteen and ends, beyond it goes on to others: the same bits
    import torch
    import fieldfare_moe as ff
    from fieldfare_moe import synthetic as syn
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rows)
    most = 32 * torch.cuda.get_device_properties(0).multi_processor_count
    ctx = ff.Context(128, 64, 16, 8, n_layers=1, max_tokens=16, act_dtype=act)
    W, S, B = syn.synth_matrix_gpu(torch, gen, most, 704)
    ids = torch.randint(0, most, (most + 17,), device="cuda", generator=gen, dtype=torch.int32)
    x = torch.randn((rows, 704), device="cuda", generator=gen).to(ctx.act)
    whole = ctx.gemv_int4_listed(W, S, B, ids, x)
    for m in (1, 16, 31, most - 15, most):
        assert torch.equal(ctx.gemv_int4_listed(W, S, B, ids[:m].contiguous(), x), whole[:, :m]), m
    ctx.close()
