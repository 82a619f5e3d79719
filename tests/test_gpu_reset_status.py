"""hs_arena_reset covers failures of the work enqueued before it."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


def test_reset_behind_a_wait_that_gives_up(hs):
    """A wait that ends at the arena's spin limit (some 50 ms) after the host has
    called the reset enqueued behind it: the reset's fills run after the failure, so
    neither status is left set and the next synchronous call succeeds."""
    import torch
    a = hs.Arena(spin_limit=1 << 15)
    try:
        word = torch.zeros(1, dtype=torch.int32, device="cuda")
        x = torch.arange(1000, dtype=torch.int32, device="cuda")
        s = torch.cuda.current_stream()
        s.synchronize()
        lib = hs.load()
        assert lib.hs_wait_value_u32(a.handle, word.data_ptr(), 1, s.cuda_stream) == 0
        a.reset(s.cuda_stream)
        st = C.c_int(-1)
        assert lib.hs_arena_device_status(a.handle, C.byref(st)) == 0 and st.value == 0
        a.sync(s.cuda_stream)  # raises if a failure is still reported
        assert hs.reduce_i32(a, x) == 499500
        # a failure with no reset behind it is reported, once
        assert lib.hs_wait_value_u32(a.handle, word.data_ptr(), 1, s.cuda_stream) == 0
        with pytest.raises(Exception):
            a.sync(s.cuda_stream)
        a.sync(s.cuda_stream)
    finally:
        a.close()
