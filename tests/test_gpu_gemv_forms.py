"""The resident matrix's GEMV where its forms meet: half a tile per block or whole tiles (by the tiles and the input rows), up to
four input rows or more. Needs a GPU: pytest -m gpu."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("m,n", [(1, 64), (16, 320), (33, 2816), (5120, 128), (5121, 704), (12288, 192), (12289, 192), (8193, 2816)])
def test_gemv_forms_agree(m, n, act):
    import torch
    import fieldfare_moe as ff
    from fieldfare_moe import synthetic as syn
    gen = torch.Generator(device="cuda")
    gen.manual_seed(m + n)
    ctx = ff.Context(128, 64, 16, 8, n_layers=1, max_tokens=16, act_dtype=act)
    W, S, B = syn.synth_matrix_gpu(torch, gen, m, n)
    mx = ctx.matrix(W, S, B)
    x = torch.randn((16, n + 8), device="cuda", generator=gen).to(ctx.act)[:, :n]      # (rows that are not dense)
    q = torch.stack((W & 15, W >> 4), 2).view(m, n).double()
    s, b = (t.double().repeat_interleave(64, 1) for t in (S, B))
    want = x.double() @ (q * s + b).T
    # A group's sum holds 64 products of x with offset + q (at most 1,039 in FP16, 143 in bf16) in fp32, then a scale and a bias per group
    # and the four slices: no more roundings than that on any path, each of 2^-24 (one bit more where the matrix unit truncates)
    # of no more than the magnitudes' sum.
    offset = 1024 if act == "fp16" else 128
    size = x.double().abs() @ ((2 * offset + q) * s + b.abs()).T
    bound = size * 2.0 ** -23 * (64 + 2 * (n // 64) + 3)
    # That is the worst case, a third of an output in FP16; errors that do not conspire are the rounding of sums that hold offset + 8 (the
    # nibbles' mean) beside nibbles that spread by 4.6, a few at a time: four such units of 2^-24, 5.4e-5 in FP16 and 7e-6 in bf16, in the 2-norm.
    usual = 4 * (offset + 8) / 4.6 * 2.0 ** -24
    rows16 = {}
    for rows in (16, 5, 4, 3, 1):
        y = mx.gemv(x[:rows], f32_out=True)
        assert ((y.double() - want[:rows]).abs() <= bound[:rows]).all(), rows
        assert (y.double() - want[:rows]).norm() <= usual * want[:rows].norm(), rows
        rows16[rows] = y
        out = torch.full((rows, m + 5), float("nan"), device="cuda").to(ctx.act)
        mx.gemv(x[:rows], out=out[:, :m])
        assert torch.equal(out[:, :m], y.to(ctx.act)) and out[:, m:].isnan().all()
        assert torch.equal(y, rows16[16][:rows]), rows         # whatever the form, a row's bits are the same
    ctx.close()
