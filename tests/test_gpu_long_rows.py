"""The forms that split long rows of logits over many blocks (sampled and greedy choice) and the matrix-unit form of the
reference-layout GEMV, at the edges of their ranges, against the CPU oracle. Needs a GPU: pytest -m gpu."""
import numpy as np
import pytest

from helpers import bf16_tensor, rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch
    assert torch.cuda.is_available()
    return torch


@pytest.fixture(scope="module")
def ctx(torch):
    import fieldfare_moe as ff
    c = ff.Context(128, 64, 16, 8, n_layers=1, max_tokens=16)
    yield c
    c.close()


# the last count of the one-block form and the first of the other, a last segment of one entry, one group more or less
@pytest.mark.parametrize("count,top_k,top_p", [(4095, 0, 1.0), (4096, 0, 1.0), (8193, 0, 1.0), (8191, 64, 0.9), (8192, 64, 0.9),
                                               (32768, 256, 0.95), (4097, 1, 1.0), (34817, 8, 1.0), (65599, 200, 1.0)])
def test_sampled_choice_at_the_edges_of_the_split_form(ctx, oracle, torch, count, top_k, top_p):
    rng = np.random.default_rng(count + top_k)
    rows = rng.normal(0, 4, (6, count)).astype(np.float32)
    rows[1] = np.round(rows[1])                                # ties at the top_k edge, over many groups
    rows[2, :] = -1.25                                         # more ties than the candidate lists hold
    rows[3, 3:] = np.nan                                       # fewer finite entries than top_k, in one group
    rows[4] = np.sort(rows[4])                                 # every survivor in the last groups
    rows[5, :] = -np.inf
    logits = torch.from_numpy(rows).cuda()
    want_tok, want_prob, gap = oracle.sample_rows(rows, 0.9, top_p, top_k, key_base=5, softcap=30.0, seed=11)
    tok, prob = ctx.sample_rows(logits, 0.9, 30.0, 11, key_base=5, top_k=top_k, top_p=top_p)
    tok, prob = tok.cpu().numpy().astype(np.uint32), prob.cpu().numpy().astype(np.float64)
    clear = gap > 1e-4                                         # log and tanh of the two machines differ by less
    assert clear.sum() >= 5 and np.array_equal(tok[clear], want_tok[clear]), (tok, want_tok, gap)
    # exp of a difference of capped logits (|c| <= 30: 2^-24 * 30 * 2 absolute each) over a sum of `count` positive terms
    same = tok == want_tok
    assert (np.abs(prob[same] - want_prob[same]) <= 1e-5 + 2e-3 * want_prob[same]).all(), (prob, want_prob)


# what the groups' largest have in common: all bits, all but the last, all but the sign and more, a whole row in one group
@pytest.mark.parametrize("count", [16384, 65536, 65600])
def test_sampled_choice_where_group_maxima_share_their_bits(ctx, oracle, torch, count):
    rng = np.random.default_rng(count)
    rows = np.full((5, count), -9.0, np.float32)
    rows[0, ::64] = 2.5
    rows[1, ::64] = np.where(rng.random((count + 63) // 64) < 0.5, np.float32(2.5), np.nextafter(np.float32(2.5), np.float32(3)))
    rows[2, ::64] = rng.choice(np.float32([-1.5, 1.5]), (count + 63) // 64)
    rows[3, :] = -np.inf
    rows[3, 640:660] = rng.normal(0, 2, 20)
    rows[4, ::64] = np.float32(2.0) + rng.random((count + 63) // 64).astype(np.float32) * np.float32(0.01)
    want_tok, want_prob, gap = oracle.sample_rows(rows, 0.9, 0.9, 48, key_base=7, softcap=30.0, seed=3)
    tok, prob = ctx.sample_rows(torch.from_numpy(rows).cuda(), 0.9, 30.0, 3, key_base=7, top_k=48, top_p=0.9)
    tok, prob = tok.cpu().numpy().astype(np.uint32), prob.cpu().numpy().astype(np.float64)
    clear = gap > 1e-4                                         # log and tanh of the two machines differ by less
    assert clear.sum() >= 4 and np.array_equal(tok[clear], want_tok[clear]), (tok, want_tok, gap)
    # (as above)
    same = tok == want_tok
    assert (np.abs(prob[same] - want_prob[same]) <= 1e-5 + 2e-3 * want_prob[same]).all(), (prob, want_prob)


@pytest.mark.parametrize("count", [1, 1023, 8192, 8193, 10241, 262144])
def test_greedy_choice_over_long_rows(ctx, oracle, torch, count):
    rng = np.random.default_rng(count)
    rows = rng.normal(0, 3, (5, count)).astype(np.float32)
    rows[1, :] = 2.0                                           # all equal: position 0
    rows[2, :] = np.nan                                        # nothing finite
    rows[3, count - 1] = 99.0                                  # the last entry wins
    rows[4, : count // 2] = np.inf
    logits = torch.from_numpy(rows).cuda()
    for cap in (0.0, 30.0):
        pos, conf = ctx.argmax_rows(logits, softcap=cap)
        want_pos, want_conf = oracle.greedy_choice_rows(rows, cap)
        assert np.array_equal(pos.cpu().numpy().astype(np.uint32), want_pos.astype(np.uint32))
        assert np.abs(conf.cpu().numpy() - want_conf).max() <= 1e-5
        assert np.array_equal(ctx.argmax_rows(logits, softcap=cap, want_conf=False).cpu().numpy(), pos.cpu().numpy())


# tiles of 16 rows: one, one and a bit, more blocks than the grid holds; one group, a K-slice of two groups, the widest row
@pytest.mark.parametrize("m,n,rows,off", [(1, 64, 1, 0), (17, 64, 16, 2), (33, 448, 3, 0), (8209, 192, 5, 0), (47, 2816, 16, 2),
                                          (31, 2752, 9, 4), (20, 2880, 2, 0)])
def test_reference_layout_gemv_at_the_edges(ctx, oracle, torch, m, n, rows, off):
    g = oracle.seed_tree_key(m + n, f"gemv-edges-{rows}")
    W, S, B = oracle.quantize_int4(g.uniform(-0.5, 0.5, m * n).reshape(m, n))
    xb = oracle.bf16_bits(g.uniform(-1.0, 1.0, rows * (n + 8))).reshape(rows, n + 8)
    raw = torch.from_numpy(np.concatenate([np.zeros(off, np.uint8), W.ravel()])).cuda()
    Sd, Bd = (torch.from_numpy(a.view(np.int16)).cuda() for a in (S, B))
    for start in (0, 1):                                       # 16-byte aligned input rows, and 2-byte aligned ones
        x = bf16_tensor(torch, xb)[:, start:start + n]
        y = ctx.gemv_int4(raw, Sd, Bd, x, f32_out=True, w_byte_offset=off).cpu().numpy()
        for r in range(rows):
            ref = oracle.gemv_int4_ref(W, S, B, oracle.bf16_to_float(xb[r, start:start + n]))
            # the offset form's sums are about 17 times the result's terms, 64 roundings of 2^-24 per group
            assert rel_err(y[r], ref) < 1e-4, (start, r)
            one = ctx.gemv_int4(raw, Sd, Bd, x[r:r + 1], f32_out=True, w_byte_offset=off).cpu().numpy()[0]
            assert np.array_equal(one.view(np.uint32), y[r].view(np.uint32))
        ids = np.array([m - 1, 0, m // 2, 0], np.int32)
        if off == 0:
            listed = ctx.gemv_int4_listed(raw, Sd, Bd, torch.from_numpy(ids).cuda(), x).cpu().numpy()
            assert np.array_equal(listed.view(np.uint32), y[:, ids].view(np.uint32))


@pytest.mark.parametrize("view", ["host address", "end of the buffer"])
def test_weight_offsets_have_the_width_of_a_pointer(ctx, oracle, torch, view):
    # gemv_int4's w_byte_offset counts from W's first byte: as far as from an address on the host to the weights on the GPU (some
    # 2^46 either way), and backwards from a view that starts behind the weights
    m, n = 33, 128
    g = oracle.seed_tree_key(0x0FF, "gemv-offset")
    W, S, B = oracle.quantize_int4(g.uniform(-0.5, 0.5, m * n).reshape(m, n))
    x = bf16_tensor(torch, oracle.bf16_bits(g.uniform(-1.0, 1.0, n)).reshape(1, n))
    raw = torch.from_numpy(np.concatenate([W.ravel(), np.zeros(64, np.uint8)])).cuda()
    Sd, Bd = (torch.from_numpy(a.view(np.int16)).cuda() for a in (S, B))
    base = torch.zeros(16, dtype=torch.uint8) if view == "host address" else raw[W.size:]
    off = raw.data_ptr() - base.data_ptr()
    assert abs(off) > (1 << 32) or view != "host address"
    y = ctx.gemv_int4(base, Sd, Bd, x, f32_out=True, w_byte_offset=off)
    assert torch.equal(y, ctx.gemv_int4(raw, Sd, Bd, x, f32_out=True))


def _choices(ctx, logits, key):
    return [t.clone() for t in (*ctx.sample_rows(logits, 0.9, 30.0, 11, key_base=key, top_k=64, top_p=0.9),
                                *ctx.sample_rows(logits, 0.9, 30.0, 11, key_base=key), *ctx.argmax_rows(logits, softcap=30.0))]


def test_captured_choices_replay_beside_eager_calls(ctx, torch):
    # a captured choice over long rows uses nothing of the context: its replays on one stream and the context's eager choices on
    # another, over other rows and in no order, leave what each leaves alone
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    mine, other = (4 * torch.randn((8, 262143), device="cuda", generator=gen) for _ in range(2))
    want, want_other = _choices(ctx, mine, 7), _choices(ctx, other, 900)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        captured = _choices(ctx, mine, 7)
    eager = []
    for replay in range(12):
        with torch.cuda.stream(side):
            graph.replay()
        eager += [_choices(ctx, other, 900) for _ in range(3)]
        if replay % 3 == 2:
            torch.cuda.synchronize()
            for got in eager:
                assert all(torch.equal(a, b) for a, b in zip(got, want_other))
            eager.clear()
            for i, (got, alone) in enumerate(zip(captured, want)):
                # positions the same; a probability is a sum in another order over up to 262,143 terms
                assert torch.equal(got, alone) if i % 2 == 0 else torch.allclose(got, alone, rtol=1e-4, atol=1e-7), (replay, i)
            for got in captured:
                got.zero_()


def test_a_captured_choice_is_one_kernel(ctx, torch):
    # the split form's two launches meet in the context's scratch; under capture there is one launch per call and no meeting
    import ctypes as C
    hip = C.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line))
    logits = torch.zeros((2, 32768), device="cuda")
    side = torch.cuda.Stream()
    for call in (lambda: ctx.sample_rows(logits, 0.9, 30.0, 11, top_k=64, top_p=0.9), lambda: ctx.sample_rows(logits, 0.9, 30.0, 11),
                 lambda: ctx.argmax_rows(logits, softcap=30.0)):
        call()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(graph, stream=side):
            call()
        nodes = C.c_size_t()
        assert hip.hipGraphGetNodes(C.c_void_p(graph.raw_cuda_graph()), None, C.byref(nodes)) == 0
        assert nodes.value == 1


def test_choices_that_need_no_scratch_order_no_streams(ctx, torch):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(6)
    long_rows, short = torch.randn((1, 16384), device="cuda", generator=gen), torch.randn((2, 1024), device="cuda", generator=gen)
    big = torch.zeros((8192, 8192), dtype=torch.bfloat16, device="cuda")
    out = torch.empty_like(big)
    # several quick streams: one of them may share the busy stream's hardware queue, all do not
    busy, quick = torch.cuda.Stream(), [torch.cuda.Stream() for _ in range(6)]
    torch.mm(big, big, out=out)
    for q in quick:
        with torch.cuda.stream(q):
            _choices(ctx, short, 1)
    torch.cuda.synchronize()
    with torch.cuda.stream(busy):
        _choices(ctx, long_rows, 1)                            # the context's scratch is this stream's
        for _ in range(150):
            torch.mm(big, big, out=out)
        end = torch.cuda.Event()
        end.record()
    done = [torch.cuda.Event() for _ in quick]
    for q, event in zip(quick, done):
        with torch.cuda.stream(q):
            _choices(ctx, short, 1)
            event.record()
    early = 0
    while not end.query():
        early = sum(event.query() for event in done)
    assert early, "the short rows waited for the other stream's work"
    torch.cuda.synchronize()


@pytest.mark.parametrize("count", [2, 63, 64, 65, 127, 1025, 1088, 1089, 2049, 7168, 7169])
def test_greedy_choice_where_waves_run_out(ctx, oracle, torch, count):
    # rows whose last values only some of a block's waves have, and those only some lanes
    rng = np.random.default_rng(count)
    rows = rng.normal(0, 3, (4, count)).astype(np.float32)
    rows[1, count - 1] = 50.0
    rows[2, : count - 1] = np.nan
    rows[3, :] = -np.inf
    logits = torch.from_numpy(rows).cuda()
    for cap in (0.0, 30.0):
        want_pos, want_conf = oracle.greedy_choice_rows(rows, cap)
        pos, conf = ctx.argmax_rows(logits, softcap=cap)
        assert np.array_equal(pos.cpu().numpy().astype(np.uint32), want_pos.astype(np.uint32))
        assert np.abs(conf.cpu().numpy() - want_conf).max() <= 1e-5
        assert np.array_equal(ctx.argmax_rows(logits, softcap=cap, want_conf=False).cpu().numpy(), pos.cpu().numpy())
