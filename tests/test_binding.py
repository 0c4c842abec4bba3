"""The native half of the Python binding, without a GPU: what it makes of its arguments before the first use of the device."""
import pytest


@pytest.fixture(scope="module")
def native():
    import fieldfare_moe as ff
    ff.lib()
    return ff._native


def _gemv_int4(native, offset):
    import torch
    w, s = torch.zeros(32, dtype=torch.uint8), torch.zeros((1, 1), dtype=torch.int16)
    return native.gemv_int4(None, w, s, s, torch.zeros((1, 64), dtype=torch.bfloat16), False, offset, torch.bfloat16)


@pytest.mark.parametrize("offset,error", [(1 << 63, OverflowError), (-(1 << 63) - 1, OverflowError), (1.0, TypeError), (None, TypeError)])
def test_a_byte_offset_is_taken_whole_or_refused(native, offset, error):
    with pytest.raises(error):
        _gemv_int4(native, offset)


def test_errors_keep_the_types_torch_gives_them(native):
    import torch
    flat = torch.zeros(64, dtype=torch.bfloat16)              # one dimension where rows are wanted
    with pytest.raises(IndexError):
        native.gemv_int4_listed(None, flat, flat, flat, flat, flat)


def test_ranks_are_the_methods_own(native):
    import torch
    rows = torch.zeros((2, 64), dtype=torch.bfloat16)
    for gate in (rows[0], rows[None]):
        with pytest.raises(ValueError):
            native.gelu_mul(None, gate, gate, gate)
    for partials in (rows, rows[None, None]):
        with pytest.raises(ValueError):
            native.reduce_token_major(None, partials, rows, torch.bfloat16)


@pytest.mark.skipif("__import__('torch').cuda.is_available()", reason="on the CPU the call ends at the device, past its arguments")
def test_setup_outputs_may_come_in_any_container(native):
    # three tensors in a sequence or one tensor of three: both get as far as the device; two do not
    import torch
    h = torch.zeros((2, 64), dtype=torch.bfloat16)
    setup = lambda out: native.post_attn_setup(None, h, h, h[0], h[0], h[0], 1e-6, 64, out, torch.bfloat16)
    for out in ((h, h, h), [h, h, h], torch.zeros((3, 2, 64), dtype=torch.bfloat16), {0: h, 1: h, 2: h}):
        with pytest.raises(RuntimeError, match="(?i)no .*(device|gpu)"):
            setup(out)
    for out, error in (((h, h), IndexError), ((h, h, 3), TypeError)):
        with pytest.raises(error):
            setup(out)
