"""The prefill's combining of a token's routes, for every top_k: the un-weighted rows added by fma in rank order, bit for bit, and
nothing of the routes that the sort drops, whatever their places in the scratch hold. Needs a GPU: pytest -m gpu."""
import numpy as np
import pytest

from helpers import make_layer, to_ff_offsets

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act", ["bf16", "fp16"])
@pytest.mark.parametrize("top_k", range(1, 9))
def test_combine_against_the_routes_rows(oracle, act, top_k):
    import torch
    import fieldfare_moe as ff
    ff.lib()
    d, f, e, t = 320, 64, 11, 77                    # 40 pieces of 16 bytes per row: tokens begin inside blocks and waves
    rng, pool, _ = make_layer(oracle, 91 + top_k, d, f, e, align=1)
    ctx = ff.Context(d, f, e, top_k, n_layers=1, max_tokens=t, act_dtype=act)
    try:
        ctx.upload_layer(0, pool.bytes, pool.stride, to_ff_offsets(ff, pool.offsets))
        dt = torch.bfloat16 if act == "bf16" else torch.float16
        x = torch.from_numpy(rng.normal(0, 1, (t, d)).astype(np.float32)).to(dt).cuda()
        idx = np.argsort(rng.random((t, e)), axis=1)[:, :top_k].astype(np.uint32)
        w = torch.from_numpy(rng.uniform(-1.0, 1.0, (t, top_k)).astype(np.float32)).to(dt)
        to = lambda a: torch.from_numpy(np.ascontiguousarray(a).view(np.int32)).cuda()
        # every route's row, from the pair list in expert order
        tok, rank = np.meshgrid(np.arange(t, dtype=np.uint32), np.arange(top_k, dtype=np.uint32), indexing="ij")
        pairs = np.stack((tok, idx, rank, np.zeros_like(idx)), -1).reshape(-1, 4)
        pairs = pairs[np.argsort(pairs[:, 1], kind="stable")]
        partials = torch.zeros((t, top_k, d), device="cuda", dtype=dt)
        ctx.prefill_pairs(0, x, to(pairs), t, partials)
        rows, weights = partials.double().cpu().numpy(), w.double().numpy()
        for share in (0.0, 0.1, 0.6, 1.0):
            lost = rng.random((t, top_k)) < share
            ctx.prefill(0, torch.full_like(x, float("nan")), to(idx), w.cuda())        # NaN in every row of the scratch
            # half of them by a zero of either sign, half by an expert that there is not
            how = rng.integers(0, 3, (t, top_k))
            wl = torch.where(torch.from_numpy(lost & (how == 0)), 0.0, torch.where(torch.from_numpy(lost & (how == 1)), -0.0, w.float())).to(dt)
            il = np.where(lost & (how == 2), np.uint32(e + 5), idx)
            y = ctx.prefill(0, x, to(il), wl.cuda()).cpu()
            acc = np.zeros((t, d), np.float32)
            for r in range(top_k):
                # (a product of two 16-bit values plus an fp32 sum: exact in float64 but for sums some 2^29 apart, so this is the fma)
                acc = np.where(lost[:, r, None], acc, (weights[:, r, None] * rows[:, r] + acc).astype(np.float32))
            assert torch.equal(y, torch.from_numpy(acc).to(dt)), (top_k, share)
    finally:
        ctx.close()
