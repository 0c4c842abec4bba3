"""Prefill chunks of layers with INT4 weight scales from 2^104 up: what a form that carries 2^24 on the scale would turn into
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


def _layer(oracle, seed, act):
    rng = np.random.default_rng(seed)
    tiny = act == "bf16"            # (FP16 has neither such weights nor such inputs)
    parts = [tuple(_part(oracle, rng, rows, cols, tiny and cols == D) for rows, cols in ((F, D), (F, D), (D, F))) for _ in range(E)]
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
