"""The second pass of the prompt router (pinned sums of the candidates, the select among them) against the pinned form of all logits, over
its forms: four, two and one wave per token, one to four 1,024-wide steps with a last one of one to four pieces, few and many ranks. Needs a GPU: pytest -m gpu."""
import numpy as np
import pytest

from helpers import bits_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("t,d,e,k", [(300, 256, 128, 8), (770, 1024, 32, 1), (1540, 1280, 64, 4), (300, 1536, 128, 5), (900, 2048, 96, 8),
                                     (1600, 2816, 128, 8), (500, 2816, 48, 4), (769, 3072, 128, 7), (300, 3328, 128, 2), (1537, 4096, 80, 8)])
def test_routes_and_weights_of_the_pinned_form(oracle, act, t, d, e, k):
    import torch
    import fieldfare_moe as ff
    ff.lib()
    rng = np.random.default_rng(d + t)
    router = rng.normal(0, 0.02, (e, d)).astype(np.float32)
    router[e - 1], router[e // 2], router[1] = router[3], router[3], router[0]      # ties: the lower index first
    bits = oracle.bf16_bits(router)
    bits[9] = bits[8]
    bits[9, d - 1] ^= 1                                                             # one bf16 step apart
    x = rng.normal(0, 1, (t, d)).astype(np.float32)
    x[1], x[2] = 0.0, x[2, 0]
    x[3], x[4] = router[3] * 50, -router[8] * 50
    x[5] *= 1e-3
    x[6, d - 1], x[7, 0], x[8, 5] = np.inf, np.nan, -np.inf
    x = torch.from_numpy(x).to(torch.bfloat16 if act == "bf16" else torch.float16).cuda()
    ctx = ff.Context(d, 64, e, k, n_layers=1, max_tokens=t, act_dtype=act)
    try:
        ctx.upload_router_bf16(0, bits)
        idx, w = ctx.router(0, x)
        want_idx, want_w, _ = ctx.router(0, x, want_logits=True)
        assert np.array_equal(idx.cpu().numpy(), want_idx.cpu().numpy())
        assert np.array_equal(bits_of(w), bits_of(want_w))
    finally:
        ctx.close()
