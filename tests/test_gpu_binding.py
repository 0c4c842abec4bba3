"""The native half of the Python binding where it meets the device: errors and threads. Needs a GPU: pytest -m gpu."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture()
def ctx():
    import fieldfare_moe as ff
    c = ff.Context(128, 64, 16, 8, n_layers=1, max_tokens=16)
    yield c
    c.close()


def test_a_failed_allocation_is_torch_s_own_error(ctx):
    # the output of 16 x 2^28 fp32 values is refused by the allocator's own limit; nothing is launched
    import torch
    w = torch.zeros(32, dtype=torch.uint8, device="cuda")
    s = torch.zeros((1, 1), dtype=torch.int16, device="cuda").expand(1 << 28, 1)
    x = torch.zeros((16, 64), dtype=torch.bfloat16, device="cuda")
    torch.cuda.set_per_process_memory_fraction(0.02)
    try:
        with pytest.raises(torch.cuda.OutOfMemoryError):
            ctx.gemv_int4(w, s, s, x, f32_out=True)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)


def test_a_call_that_waits_lets_other_threads_run(ctx):
    # with profiling on a call waits for its kernel, here behind some 100 ms of products: the other thread's clock goes on
    import threading
    import time
    import numpy as np
    import torch
    rng = np.random.default_rng(0)
    mx = ctx.matrix(rng.integers(0, 256, (64, 64), dtype=np.uint8), *(np.full((64, 2), 0x3C00, np.uint16) for _ in range(2)))
    x = torch.zeros((1, 128), dtype=torch.bfloat16, device="cuda")
    big = torch.zeros((8192, 8192), dtype=torch.bfloat16, device="cuda")
    out = torch.empty_like(big)
    ctx.set_profiling(True)
    mx.gemv(x)
    torch.mm(big, big, out=out)
    torch.cuda.synchronize()
    stamps, stop = [], threading.Event()

    def clock():
        while not stop.is_set():
            stamps.append(time.perf_counter())
            time.sleep(0.001)

    for _ in range(150):
        torch.mm(big, big, out=out)
    th = threading.Thread(target=clock)
    th.start()
    time.sleep(0.005)
    begin = time.perf_counter()
    mx.gemv(x)
    end = time.perf_counter()
    stop.set()
    th.join()
    inside = [begin] + [s for s in stamps if begin < s < end] + [end]
    assert end - begin > 0.02, "the call did not wait"
    assert max(b - a for a, b in zip(inside, inside[1:])) < 0.5 * (end - begin)
    mx.close()


def test_setup_outputs_in_one_tensor(ctx):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    hidden, attn = (torch.randn((5, 128), device="cuda", generator=g).to(torch.bfloat16) for _ in range(2))
    w = [torch.rand(128, device="cuda", generator=g).to(torch.bfloat16) for _ in range(3)]
    out = torch.zeros((3, 5, 128), dtype=torch.bfloat16, device="cuda")
    want = ctx.post_attn_setup(hidden.clone(), attn, *w)
    assert ctx.post_attn_setup(hidden.clone(), attn, *w, out=out) is out
    assert all(torch.equal(a, b) for a, b in zip(out, want))
