"""Matrices and layers of more bytes than the memory side's cache holds: their weights are read with another cache hint, in kernels of
their own. Same bits as the forms without it. Needs a GPU: pytest -m gpu."""
import pytest

pytestmark = pytest.mark.gpu

# 262,144 rows in 4 bits, 131,072 in 8: 277 MB at 2,112 columns, where 4 bits are read so for up to four rows, and 294 MB at 2,240
@pytest.mark.parametrize("N", [2112, 2240])
@pytest.mark.parametrize("act", ["bf16", "fp16"])
def test_rows_of_a_large_matrix(act, N):
    import torch
    import fieldfare_moe as ff
    from fieldfare_moe import synthetic as syn
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    dt = torch.bfloat16 if act == "bf16" else torch.float16
    ctx = ff.Context(256, 128, 8, 8, n_layers=1, max_tokens=16, act_dtype=act)
    try:
        m = 262144
        parts = syn.synth_matrix_gpu(torch, gen, m, N)
        head = ctx.matrix(*parts, greedy=True)
        x = torch.randn((16, N), device="cuda", generator=gen).to(dt)
        at = torch.tensor([0, 31, 32, 4097, 131071, 200000, m - 33, m - 1], device="cuda")
        few = ctx.matrix(*[p[at].contiguous() for p in parts])
        for rows in (1, 4, 5, 16):
            y = head.gemv(x[:rows], f32_out=True)
            assert torch.equal(y[:, at], few.gemv(x[:rows], f32_out=True))
            assert torch.equal(head.gemv(x[:rows])[:, at], few.gemv(x[:rows]))
            best, conf = head.greedy_conf(x[:rows], softcap=30.0)
            assert torch.equal(best.to(torch.int64), y.argmax(1))
            # the winner's share of the capped logits' softmax: an exponential's argument is off by some units of 2^-24 of 60 (two caps of
            # at most 30), 2e-5, and a sum of positive values by a unit for each of the few hundred that one place adds up, 4e-5
            capped = 30.0 * torch.tanh(y.double() / 30.0)
            want = torch.softmax(capped, 1).gather(1, best.to(torch.int64)[:, None])[:, 0]
            assert ((conf.double() - want).abs() <= 1e-4 * want).all(), rows
    finally:
        ctx.close()


@pytest.mark.parametrize("act", ["bf16", "fp16"])
def test_rows_of_a_large_8bit_matrix(act, N=2112):
    import torch
    import fieldfare_moe as ff
    gen = torch.Generator(device="cuda")
    gen.manual_seed(8)
    dt = torch.bfloat16 if act == "bf16" else torch.float16
    ctx = ff.Context(256, 128, 8, 8, n_layers=1, max_tokens=16, act_dtype=act)
    try:
        m = 131072
        w = torch.randint(0, 256, (m, N), dtype=torch.uint8, device="cuda", generator=gen)
        s = (torch.randn((m, N // ff.GROUP), device="cuda", generator=gen) * 0.001).abs().to(torch.bfloat16)
        b = (-128.0 * s.float() + torch.randn((m, N // ff.GROUP), device="cuda", generator=gen) * 1e-3).to(torch.bfloat16)
        x = torch.randn((16, N), device="cuda", generator=gen).to(dt)
        at = torch.tensor([0, 15, 16, 4097, 65535, 100000, m - 17, m - 1], device="cuda")
        large = ctx.matrix_int8(w, s, b)
        few = ctx.matrix_int8(*[p[at].contiguous() for p in (w, s, b)])
        scale, bias = (p[at].double().repeat_interleave(ff.GROUP, 1) for p in (s, b))
        want = x.double() @ (scale * w[at].double() + bias).T
        for rows in (1, 4, 5, 16):
            y = large.gemv(x[:rows], f32_out=True)
            assert torch.equal(y[:, at], few.gemv(x[:rows], f32_out=True))
            assert torch.equal(large.gemv(x[:rows])[:, at], few.gemv(x[:rows]))
            # (the nibbles enter as 128 + q, 1024 + q in FP16, and spread by 4.6: four roundings of such a sum)
            usual = 4 * ((1024 if act == "fp16" else 128) + 8) / 4.6 * 2.0 ** -24
            assert (y[:, at].double() - want[:rows]).norm() <= usual * want[:rows].norm(), rows
    finally:
        ctx.close()


@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("layers", [1, 2])
def test_short_chunk_of_a_large_layer(act, layers):
    # 128 experts of 2,816 x 704 (80 of them fill the memory side's cache, 40 where the context has two layers): a chunk that reaches
    # them all, or 30, or 60, beside parts of it that could not reach as many as the cache holds
    import torch
    import fieldfare_moe as ff
    from fieldfare_moe import synthetic as syn
    gen = torch.Generator(device="cuda")
    gen.manual_seed(6)
    ctx = ff.Context(syn.D, syn.F, syn.E, syn.K, n_layers=layers, max_tokens=512, act_dtype=act)
    try:
        offsets, _ = syn.layout_offsets(syn.D, syn.F, align=16)
        for layer in range(layers):
            ctx.upload_layer(layer, syn.synth_layer_gpu(torch, gen, offsets).view(-1), syn.STRIDE, offsets)
        dt = torch.bfloat16 if act == "bf16" else torch.float16
        for t in (40, 301, 500):                    # tiles of 16 (bf16), 32 and 64 pairs; one expert with whole tiles
            x = torch.randn((t, syn.D), device="cuda", generator=gen).to(dt)
            for live in (syn.E, 60, 30):
                idx = torch.topk(torch.rand((t, live), device="cuda", generator=gen), syn.K, dim=1).indices.to(torch.int32)
                idx[:, 0] = torch.where((idx[:, 1:] == 7).any(1), idx[:, 0], 7)
                idx = (idx * (syn.E // live)).contiguous()
                w = (torch.rand((t, syn.K), device="cuda", generator=gen) * 0.2 + 0.05).to(dt)
                y = ctx.prefill(layers - 1, x, idx, w)
                n_pairs, _, counts = ctx.prefill_stats()
                assert n_pairs == t * syn.K and (counts > 0).sum() == len(torch.unique(idx))
                for part in (slice(0, 2), slice(t - 3, t)):
                    assert torch.equal(ctx.prefill(layers - 1, x[part].contiguous(), idx[part].contiguous(), w[part].contiguous()), y[part])
    finally:
        ctx.close()


@pytest.mark.parametrize("act", ["bf16", "fp16"])
def test_whole_and_lone_tiles_of_a_large_layer(act):
    # experts whose pairs are one short, one whole, two whole and a whole and a short tile of 32, in a layer read once and in calls of
    # few of its experts, whose tiles are the others' too
    import torch
    import fieldfare_moe as ff
    from fieldfare_moe import synthetic as syn
    gen = torch.Generator(device="cuda")
    gen.manual_seed(7)
    ctx = ff.Context(syn.D, syn.F, syn.E, 1, n_layers=1, max_tokens=4096, act_dtype=act)
    try:
        offsets, _ = syn.layout_offsets(syn.D, syn.F, align=16)
        ctx.upload_layer(0, syn.synth_layer_gpu(torch, gen, offsets).view(-1), syn.STRIDE, offsets)
        counts = torch.tensor([(1, 31, 32, 33, 64, 16, 3, 0)[e % 8] for e in range(syn.E)])
        t = int(counts.sum())
        assert t <= 28 * syn.E                      # tiles of 32
        idx = torch.repeat_interleave(torch.arange(syn.E), counts).to(torch.int32)[torch.randperm(t)].cuda()[:, None].contiguous()
        dt = torch.bfloat16 if act == "bf16" else torch.float16
        x = torch.randn((t, syn.D), device="cuda", generator=gen).to(dt)
        w = (torch.rand((t, 1), device="cuda", generator=gen) * 0.2 + 0.05).to(dt)
        y = ctx.prefill(0, x, idx, w)
        for some in range(16):                      # eight experts at a time, one of each count
            at = torch.nonzero(idx[:, 0] // 8 == some)[:, 0]
            assert torch.equal(ctx.prefill(0, x[at].contiguous(), idx[at].contiguous(), w[at].contiguous()), y[at]), some
    finally:
        ctx.close()
