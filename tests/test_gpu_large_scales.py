"""Prefill and dense chunks of layers with weight scales from 2^104 up: what a form that carries 2^24 on the scale would turn into
infinities and NaN is as finite here as q * scale + bias is - whole groups with q = 0 under such a scale (their weights are the
biases), and in bf16 groups whose inputs are as small as the scale is large. Needs a GPU: pytest -m gpu."""
import numpy as np
import pytest

from helpers import to_ff_offsets
from test_gpu_prefill_gemm import _check

pytestmark = pytest.mark.gpu

D, F, E = 320, 192, 4
TINY = slice(64, 128)               # columns of the inputs that are near 2^-112 in bf16


def _part(oracle, rng, rows, cols, tiny):
    """Ordinary weights, but: in every third row group 0 is q = 0 under scales of 2^104 .. 2^126; with `tiny` in every third row
    group 1 has scales of 2^104 .. 2^112 and any q."""
    W = rng.integers(0, 256, size=(rows, cols // 2), dtype=np.uint8)
    scale = np.abs(rng.normal(0, 0.01, size=(rows, cols // 64))).astype(np.float32)
    bias = -8.0 * oracle.bf16_to_float(oracle.bf16_bits(scale)) + rng.normal(0, 1e-3, size=scale.shape).astype(np.float32)
    some = np.arange(0, rows, 3)
    W[some, :32] = 0
    scale[some, 0] = np.exp2(104.0 + some % 23)
    bias[some, 0] = rng.normal(0, 0.02, size=len(some))
    if tiny:
        some = np.arange(1, rows, 3)
        scale[some, 1] = np.exp2(104.0 + some % 9)
        bias[some, 1] = -8.0 * scale[some, 1]
    return W, oracle.bf16_bits(scale), oracle.bf16_bits(bias.astype(np.float32))


def _layer(oracle, seed, act, e=E):
    rng = np.random.default_rng(seed)
    tiny = act == "bf16"            # (FP16 has neither such weights nor such inputs)
    parts = [tuple(_part(oracle, rng, rows, cols, tiny and cols == D) for rows, cols in ((F, D), (F, D), (D, F))) for _ in range(e)]
    return rng, oracle.pool_from_parts(parts, D, F, 1, None)


def _rows(torch, rng, t, act):
    x = rng.normal(0, 1, (t, D)).astype(np.float32)
    if act == "bf16":
        x[:, TINY] = np.ldexp(rng.uniform(1, 2, (t, 64)) * rng.choice([-1.0, 1.0], (t, 64)), -112)
    return torch.from_numpy(x).to(torch.bfloat16 if act == "bf16" else torch.float16)


# 20 and 150 rows: where the streaming product serves; 260 and 1,200: the grouped GEMMs, one and two tiles per expert
@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("t", [20, 150, 260, 1200])
def test_chunks_against_the_oracle(oracle, act, t):
    import torch
    import fieldfare_moe as ff
    ff.lib()
    rng, pool = _layer(oracle, t, act)
    ctx = ff.Context(D, F, E, 1, n_layers=1, max_tokens=t, act_dtype=act)
    try:
        ctx.upload_layer(0, pool.bytes, pool.stride, to_ff_offsets(ff, pool.offsets))
        x = _rows(torch, rng, t, act)
        idx = rng.integers(0, E, (t, 1)).astype(np.uint32)
        w = torch.from_numpy(rng.uniform(0.2, 1.0, (t, 1)).astype(np.float32)).to(x.dtype)
        y = ctx.prefill(0, x.cuda(), torch.from_numpy(idx.view(np.int32)).cuda(), w.cuda()).float().cpu().numpy()
        assert np.isfinite(y).all()
        _check(oracle, pool, E, idx, x, w, y, act)
    finally:
        ctx.close()


# a dense FFN's chunk where bands of rows serve other layers of these widths (in bf16 up to 896 rows, in FP16 up to 384) and beyond
@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("t", [17, 100, 384, 385, 640, 896, 897])
def test_dense_chunks_against_the_oracle(oracle, act, t):
    import torch
    import fieldfare_moe as ff
    ff.lib()
    rng, pool = _layer(oracle, t, act, 1)
    ctx = ff.Context(D, F, 1, 1, n_layers=1, max_tokens=t, act_dtype=act)
    try:
        ctx.upload_layer(0, pool.bytes, pool.stride, to_ff_offsets(ff, pool.offsets))
        x = _rows(torch, rng, t, act)
        y = ctx.dense_ffn(0, x.cuda()).float().cpu().numpy()
        assert np.isfinite(y).all()
        _check(oracle, pool, 1, np.zeros((t, 1), np.uint32), x, torch.ones((t, 1), dtype=x.dtype), y, act)
    finally:
        ctx.close()


def _part8(oracle, rng, rows, cols):
    """8-bit weights around a zero point of 128, but in every third row group 0 is q = 0 under scales of 2^104 .. 2^123."""
    W = rng.integers(0, 256, size=(rows, cols), dtype=np.uint8)
    scale = np.abs(rng.normal(0, 0.001, size=(rows, cols // 64))).astype(np.float32)
    bias = -128.0 * oracle.bf16_to_float(oracle.bf16_bits(scale)) + rng.normal(0, 1e-3, size=scale.shape).astype(np.float32)
    some = np.arange(0, rows, 3)
    W[some, :64] = 0
    scale[some, 0] = np.exp2(104.0 + some % 20)
    bias[some, 0] = rng.normal(0, 0.02, size=len(some))
    return W, oracle.bf16_bits(scale), oracle.bf16_bits(bias.astype(np.float32))


# 8 bits: from 192 rows on, where bf16 chunks of other layers of these widths stay in bands up to 639
@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("t", [192, 300, 512, 639, 640])
def test_8_bit_dense_chunks_against_float64(oracle, act, t):
    import torch
    import fieldfare_moe as ff
    ff.lib()
    rng = np.random.default_rng(t)
    parts = tuple(_part8(oracle, rng, rows, cols) for rows, cols in ((F, D), (F, D), (D, F)))
    dt = torch.bfloat16 if act == "bf16" else torch.float16
    x = torch.from_numpy(rng.normal(0, 1, (t, D)).astype(np.float32)).to(dt)
    ctx = ff.Context(D, F, 1, 1, n_layers=1, max_tokens=t, act_dtype=act)
    try:
        ctx.upload_expert_parts(0, 0, *parts, int8=True)
        y = ctx.dense_ffn(0, x.cuda()).double().cpu().numpy()
        g, u, dn = (oracle.dequantize_int8(*p).astype(np.float64) for p in parts)
        rnd = lambda a: torch.from_numpy(a).to(torch.float32).to(dt).double().numpy()
        gate, up = rnd(x.double().numpy() @ g.T), rnd(x.double().numpy() @ u.T)
        a = rnd(rnd(0.5 * gate * (1 + np.tanh(0.7978845608028654 * (gate + 0.044715 * gate ** 3)))) * up)
        ref, spread = a @ dn.T, np.abs(a) @ np.abs(dn.T)
        # one unit of gate, up and the activation each through the down product, where an fp32 sum near a rounding's middle goes the
        # other way; then the output's own half unit
        unit = 2.0 ** (-8 if act == "bf16" else -11)
        assert np.isfinite(y).all() and np.all(np.abs(y - ref) <= 1.1 * unit * (4 * spread + np.abs(ref)))
        # and the same layer replaced by one without such scales: the bits of a context that never had one
        plain = tuple((W, np.minimum(S, oracle.bf16_bits(np.float32([0.01]))[0]), B) for W, S, B in parts)
        ctx.upload_expert_parts(0, 0, *plain, int8=True)
        z = ctx.dense_ffn(0, x.cuda())
        other = ff.Context(D, F, 1, 1, n_layers=1, max_tokens=t, act_dtype=act)
        other.upload_expert_parts(0, 0, *plain, int8=True)
        assert torch.equal(other.dense_ffn(0, x.cuda()), z)
        other.close()
    finally:
        ctx.close()


def test_an_upload_decides_for_its_experts(oracle):
    """Experts one at a time: with one of them large the chunk is finite; replaced, it has the bits of a layer that never was."""
    import torch
    import fieldfare_moe as ff
    ff.lib()
    rng, large = _layer(oracle, 11, "fp16")
    plain = oracle.random_pool(rng, E, D, F, align=1)
    t = 260
    x, idx = _rows(torch, rng, t, "fp16").cuda(), torch.from_numpy(rng.integers(0, E, (t, 1)).astype(np.int32)).cuda()
    w = torch.ones((t, 1), dtype=torch.float16, device="cuda")

    def cuda(pool, e):
        bf = lambda a: torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).cuda().view(torch.bfloat16)
        return [(torch.from_numpy(np.ascontiguousarray(W)).cuda(), bf(S), bf(B)) for W, S, B in (pool.sub(e, n) for n in ("gate", "up", "down"))]

    ctx = ff.Context(D, F, E, 1, n_layers=1, max_tokens=t, act_dtype="fp16")
    try:
        ctx.upload_layer(0, plain.bytes, plain.stride, to_ff_offsets(ff, plain.offsets))
        want = ctx.prefill(0, x, idx, w)
        ctx.upload_expert_parts(0, 2, *cuda(large, 2))
        mixed = ctx.prefill(0, x, idx, w)
        others = (idx[:, 0] != 2).nonzero()[:, 0]
        assert torch.isfinite(mixed).all() and torch.equal(mixed[others], want[others]) and not torch.equal(mixed, want)
        ctx.upload_expert_parts(0, 2, *cuda(plain, 2))
        assert torch.equal(ctx.prefill(0, x, idx, w), want)
    finally:
        ctx.close()


@pytest.mark.parametrize("act", ["bf16", "fp16"])
def test_tile_weights_bit_for_bit(oracle, act):
    import torch
    import fieldfare_moe as ff
    ff.lib()
    _, pool = _layer(oracle, 5, act)
    ctx = ff.Context(D, F, E, 1, n_layers=1, max_tokens=16, act_dtype=act)
    try:
        ctx.upload_layer(0, pool.bytes, pool.stride, to_ff_offsets(ff, pool.offsets))
        dt = torch.bfloat16 if act == "bf16" else torch.float16
        for which, name in ((ff.GATE, "gate"), (ff.UP, "up"), (ff.DOWN, "down")):
            want = torch.from_numpy(oracle.dequantize_int4(*pool.sub(E - 1, name))).to(dt)
            assert torch.equal(ctx.prefill_tiles(0, E - 1, which).cpu().view(torch.int16), want.view(torch.int16)), name
    finally:
        ctx.close()
