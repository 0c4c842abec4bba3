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
