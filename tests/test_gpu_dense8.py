"""The 8-bit dense layer's GEMMs on integer operands (640 rows and more, wide layers from 560 or 385 on): ragged row tiles either side of the tile sizes, an
output width that fills half a block of columns, widths of an odd number of groups, both activation types, inputs with a large
common part (so that the bias columns carry most of a sum), rows that overflow. Needs a GPU: pytest -m gpu."""
import numpy as np
import pytest

from helpers import cosine, rel_err

pytestmark = pytest.mark.gpu


def _gelu(x):
    return 0.5 * x * (1 + np.tanh(0.7978845608028654 * (x + 0.044715 * x ** 3)))


@pytest.mark.parametrize("act", ["bf16", "fp16"])
# K of one group to 44, output widths of a quarter of a 256-row block to eleven blocks
@pytest.mark.parametrize("d,f,t", [(128, 64, 640), (192, 320, 641), (64, 704, 703), (192, 1472, 1088), (448, 192, 1089), (2816, 128, 1153),
                                   (192, 2816, 1025), (2112, 2112, 1217), (2816, 2112, 386), (2816, 2112, 543), (2816, 1024, 561)])
def test_rows_against_float64(oracle, act, d, f, t):
    import torch
    import fieldfare_moe as ff
    ff.lib()
    g = oracle.seed_tree_key(0x1A8, f"dense8-{d}-{f}-{t}")
    parts = tuple(oracle.quantize_int8(g.uniform(-0.2, 0.2, r * c).reshape(r, c)) for r, c in ((f, d), (f, d), (d, f)))
    dt = torch.bfloat16 if act == "bf16" else torch.float16
    x = torch.from_numpy((g.uniform(-1.0, 1.0, t * d) + 0.5).reshape(t, d).astype(np.float32)).to(dt)
    ctx = ff.Context(d, f, 1, 1, n_layers=1, max_tokens=t, act_dtype=act)
    try:
        ctx.upload_expert_parts(0, 0, *parts, int8=True)
        y = ctx.dense_ffn(0, x.cuda())
        yf = y.float().cpu().numpy()
        gw, uw, dw = (oracle.dequantize_int8(*p).astype(np.float64) for p in parts)
        xf = x.double().numpy()
        # as the layer rounds: gate and up to the activation type, the product once more, the output row
        rnd = lambda a: torch.from_numpy(a).to(torch.float32).to(dt).double().numpy()
        a = rnd(_gelu(rnd(xf @ gw.T)) * rnd(xf @ uw.T))
        ref, spread = a @ dw.T, np.abs(a) @ np.abs(dw.T)
        # where a sum falls near a rounding's middle, the fp32 sum may round the other way: one unit (2^-8 bf16, 2^-11 FP16) of
        # gate, up and the activation each (gelu' is below 1.13), through the down product; then the output's own half unit
        unit = 2.0 ** (-8 if act == "bf16" else -11)
        assert np.all(np.abs(yf - ref) <= 1.1 * unit * (4 * spread + np.abs(ref)))
        assert cosine(yf, ref) > 0.99999 and rel_err(yf, ref) < (1e-2 if act == "bf16" else 1.5e-3)
        # a row does not depend on the rows beside it (both tile sizes sum in one order)
        # from 1,024 rows on every width takes this form, those here from 640 on, wide ones from 560 or 385 on
        first = 1024 if t > 1024 else 640 if t >= 640 else 560 if d * f < 4000000 else 385
        part = ctx.dense_ffn(0, x[:first].cuda()).float().cpu().numpy()
        assert np.array_equal(part, yf[:first])
        # other rows are untouched by one that is not finite
        x[7, 3] = float("inf")
        got = ctx.dense_ffn(0, x.cuda()).float().cpu().numpy()
        assert not np.isfinite(got[7]).any() and np.array_equal(np.delete(got, 7, 0), np.delete(yf, 7, 0))
    finally:
        ctx.close()


def _parts(oracle, d, f, key):
    g = oracle.seed_tree_key(0x1A8, key)
    weights = [g.uniform(-0.2, 0.2, r * c).reshape(r, c) for r, c in ((f, d), (f, d), (d, f))]
    return g, tuple(oracle.quantize_int8(w) for w in weights), tuple(oracle.quantize_int4(w) for w in weights)


def test_the_form_follows_the_activation_type(oracle):
    # one context through both types and back, a 4-bit upload and an 8-bit one again: every state gives the bits of a context that
    # was made for it, so the operands are remade when the context changes type and go with a 4-bit upload
    import torch
    import fieldfare_moe as ff
    ff.lib()
    d, f, t = 128, 192, 650
    g, int8, int4 = _parts(oracle, d, f, "dense8-types")
    x = torch.from_numpy(g.uniform(-1.0, 1.0, t * d).reshape(t, d).astype(np.float32))
    run = lambda c, act: c.dense_ffn(0, x.to(torch.bfloat16 if act == "bf16" else torch.float16).cuda()).float().cpu().numpy()
    alone = {}
    for act in ("bf16", "fp16"):
        for bits, parts in ((8, int8), (4, int4)):
            ctx = ff.Context(d, f, 1, 1, n_layers=1, max_tokens=t, act_dtype=act)
            ctx.upload_expert_parts(0, 0, *parts, int8=bits == 8)
            alone[act, bits] = run(ctx, act)
            ctx.close()
    assert rel_err(alone["bf16", 8], alone["fp16", 8]) < 2e-2 and not np.array_equal(alone["bf16", 8], alone["fp16", 8])
    assert not np.array_equal(alone["bf16", 8], alone["bf16", 4])
    ctx = ff.Context(d, f, 1, 1, n_layers=1, max_tokens=t)
    try:
        for step, (act, upload, bits) in enumerate((("bf16", int8, 8), ("fp16", None, 8), ("bf16", None, 8), ("bf16", int4, 4), ("fp16", None, 4),
                                                    ("fp16", int8, 8), ("bf16", None, 8))):
            ctx.set_act_dtype(act)
            if upload:
                ctx.upload_expert_parts(0, 0, *upload, int8=bits == 8)
            assert np.array_equal(run(ctx, act), alone[act, bits]), (step, act, bits)
    finally:
        ctx.close()


@pytest.mark.parametrize("d,f,line", [(2816, 128, 1024), (1024, 1984, 689), (128, 192, 640), (2816, 2112, 385), (2816, 1024, 560)])
def test_the_line_to_the_library_form(oracle, d, f, line):
    # the row before and the row after the line that the widths draw, in a context for more rows and in one for the row before alone
    import torch
    import fieldfare_moe as ff
    ff.lib()
    g, int8, _ = _parts(oracle, d, f, f"dense8-line-{d}")
    x = torch.from_numpy(g.uniform(-1.0, 1.0, line * d).reshape(line, d).astype(np.float32)).to(torch.bfloat16).cuda()
    outs = []
    for cap in (line, line - 1):
        ctx = ff.Context(d, f, 1, 1, n_layers=1, max_tokens=cap)
        ctx.upload_expert_parts(0, 0, *int8, int8=True)
        outs += [ctx.dense_ffn(0, x[:t]).float().cpu().numpy() for t in (line - 1, line) if t <= cap]
        ctx.close()
    library, integers, alone = outs
    assert np.array_equal(library, alone)                    # the same form, whatever the context could also do
    assert not np.array_equal(library, integers[:-1])        # another one
    # 16-bit results of one rounding each way, of sums whose weights have 16 significant bits or all of them
    assert rel_err(library, integers[:-1]) < 2e-2 and cosine(library, integers[:-1]) > 0.9999


@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("t", [640, 1153])
def test_the_gemms_in_a_graph(oracle, act, t):
    # replayed with new rows in the input and eager calls of the context (another row count, the streaming form) in between
    import torch
    import fieldfare_moe as ff
    ff.lib()
    d, f = 192, 320
    g, int8, _ = _parts(oracle, d, f, f"dense8-graph-{t}")
    dt = torch.bfloat16 if act == "bf16" else torch.float16
    ctx = ff.Context(d, f, 1, 1, n_layers=1, max_tokens=t, act_dtype=act)
    try:
        ctx.upload_expert_parts(0, 0, *int8, int8=True)
        rows = [torch.from_numpy(g.uniform(-1.0, 1.0, t * d).reshape(t, d).astype(np.float32)).to(dt).cuda() for _ in range(4)]
        want = [ctx.dense_ffn(0, r) for r in rows]
        x, y = rows[0].clone(), torch.empty((t, d), dtype=dt, device="cuda")
        torch.cuda.synchronize()
        graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        with torch.cuda.graph(graph, stream=side):
            ctx.dense_ffn(0, x, out=y)
        for r, alone in zip(rows, want):
            x.copy_(r)
            y.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y.view(torch.int16), alone.view(torch.int16))
            ctx.dense_ffn(0, rows[1][:640])
            ctx.dense_ffn(0, rows[2][:33])
            torch.cuda.synchronize()
    finally:
        ctx.close()


@pytest.mark.parametrize("act", ["bf16", "fp16"])
# every number of 16-row blocks per tile (3 to 15) in both products, last tiles of one block and more; odd numbers of 128-row blocks
@pytest.mark.parametrize("d,f,rows", [(448, 2112, (1024, 1206, 1457, 1682, 1927, 2165, 2403, 2657, 2886, 3124, 3377)),
                                      (2112, 448, (1025, 1346, 1794, 2242, 2691, 3138, 3586, 4034, 4482, 4930, 5378, 5826)),
                                      (704, 1408, (1024, 1108)), (2816, 64, (5154,))])
def test_tiles_of_the_row_count(oracle, act, d, f, rows):
    # the largest chunk against 64-bit products (first and last rows), every other one, cut elsewhere, to the same bits
    import torch
    import fieldfare_moe as ff
    ff.lib()
    g, int8, _ = _parts(oracle, d, f, f"dense8-tiles-{d}")
    t = max(rows)
    dt = torch.bfloat16 if act == "bf16" else torch.float16
    x = torch.from_numpy((g.uniform(-1.0, 1.0, t * d) + 0.25).reshape(t, d).astype(np.float32)).to(dt)
    ctx = ff.Context(d, f, 1, 1, n_layers=1, max_tokens=t, act_dtype=act)
    try:
        ctx.upload_expert_parts(0, 0, *int8, int8=True)
        y = ctx.dense_ffn(0, x.cuda())
        some = np.r_[0:260, t - 260:t]
        gw, uw, dw = (oracle.dequantize_int8(*p).astype(np.float64) for p in int8)
        xf = x[some].double().numpy()
        rnd = lambda a: torch.from_numpy(a).to(torch.float32).to(dt).double().numpy()
        a = rnd(_gelu(rnd(xf @ gw.T)) * rnd(xf @ uw.T))
        ref, spread = a @ dw.T, np.abs(a) @ np.abs(dw.T)
        unit = 2.0 ** (-8 if act == "bf16" else -11)         # the bound of test_rows_against_float64
        assert np.all(np.abs(y[some].float().cpu().numpy() - ref) <= 1.1 * unit * (4 * spread + np.abs(ref)))
        for n in rows:
            # (after rows of NaN through the scratch and into NaN: what is not written is not equal)
            ctx.dense_ffn(0, torch.full_like(x, float("nan")).cuda())
            assert torch.equal(ctx.dense_ffn(0, x[:n].cuda(), out=torch.full_like(y[:n], float("nan"))), y[:n]), n
    finally:
        ctx.close()
