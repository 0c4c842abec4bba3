"""The native half of the Python binding where it meets the device: errors and threads. Run on the GPU box: pytest -m gpu."""
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
