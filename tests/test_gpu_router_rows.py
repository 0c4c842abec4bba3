"""Router routes of a short prompt either side of the row count from which the prefill router runs in two passes (160, less
where many experts meet few columns: after 37 at 256 x 128 and 79 at 2,048 x 128, in FP16 46 and 96; narrow tables after 4,096 rows x
experts, in FP16 5,120): the same routes and weights,
bit for bit, as the pinned sums of all logits. Needs a GPU: pytest -m gpu."""
import numpy as np
import pytest

from helpers import bf16_tensor, bits_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("d,e,t", [(2816, 128, 17), (2816, 128, 160), (2816, 128, 161), (1024, 16, 160), (4096, 128, 163),
                                   (256, 128, 73), (256, 128, 74), (256, 128, 78), (2048, 128, 150), (2048, 128, 151),
                                   (256, 128, 37), (256, 128, 38), (256, 128, 46), (256, 128, 47), (2048, 128, 79), (2048, 128, 80), (2048, 128, 96), (2048, 128, 97), (512, 32, 128), (512, 32, 129), (512, 32, 160), (512, 32, 161), (256, 16, 160)])
def test_routes_either_side_of_the_two_pass_line(oracle, act, d, e, t):
    import torch
    import fieldfare_moe as ff
    ff.lib()
    rng = np.random.default_rng(d + t)
    bits = oracle.bf16_bits(rng.normal(0, 0.02, (e, d)).astype(np.float32))
    bits[5] = bits[3]                           # exact ties: the lower index wins
    bits[9] = bits[8]
    bits[9, 17] ^= 1                            # one bf16 step apart in one element
    wf = oracle.bf16_to_float(bits)
    x = rng.normal(0, 1, (t, d)).astype(np.float32)
    last = t - 1                                # a row that a block of four has to itself or shares
    x[1] *= 1e3
    x[2] = 0.0
    x[3] = wf[3] * 50                           # the tied experts lead
    x[4, 100] = np.inf
    x[5, 5] = np.nan
    x[last] = 50.0 * (1.5 * wf[[0, 1, 2, 6, 7, 10, 11]].sum(axis=0) + wf[8])     # experts 8 and 9 at the select's edge
    xt = torch.from_numpy(x).to(torch.float16).cuda() if act == "fp16" else bf16_tensor(torch, oracle.bf16_bits(x))
    ctx = ff.Context(d, 64, e, 8, n_layers=1, max_tokens=t, act_dtype=act)
    try:
        ctx.upload_router_bf16(0, bits)
        idx, w = ctx.router(0, xt)
        idx_ref, w_ref, _ = ctx.router(0, xt, want_logits=True)
        assert np.array_equal(idx.cpu().numpy(), idx_ref.cpu().numpy())
        assert np.array_equal(bits_of(w), bits_of(w_ref))
    finally:
        ctx.close()
