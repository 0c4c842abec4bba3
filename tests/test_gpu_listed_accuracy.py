"""The listed GEMV's fp32 logits against float64: no further off than dot products on the vector unit left them (a relative
error of 8.6e-7 in bf16, 1.6e-5 in FP16 at 2,816 columns). Needs a GPU: pytest -m gpu."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act,bound", [("bf16", 8e-7), ("fp16", 1.5e-5)])
@pytest.mark.parametrize("m,n,rows", [(515, 2816, 16), (1000, 2752, 3), (300, 512, 1)])
def test_listed_logits_against_float64(oracle, act, bound, m, n, rows):
    import torch
    import fieldfare_moe as ff
    ff.lib()
    rng = np.random.default_rng(m + n)
    W, S, B = oracle.quantize_int4(rng.normal(0, 0.02, (m, n)).astype(np.float32))
    x = torch.from_numpy(rng.normal(0, 1, (rows, n)).astype(np.float32)).to(torch.bfloat16 if act == "bf16" else torch.float16)
    ids = rng.permutation(m)[: m // 2].astype(np.int32)
    ctx = ff.Context(256, 128, 8, 8, n_layers=1, max_tokens=16, act_dtype=act)
    try:
        bf = lambda a: torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).cuda().view(torch.bfloat16)
        y = ctx.gemv_int4_listed(torch.from_numpy(W).cuda(), bf(S), bf(B), torch.from_numpy(ids).cuda(), x.cuda()).double().cpu().numpy()
        ref = x.double().numpy() @ oracle.dequantize_int4(W, S, B).astype(np.float64)[ids].T
        assert np.linalg.norm(y - ref) <= bound * np.linalg.norm(ref)
    finally:
        ctx.close()
