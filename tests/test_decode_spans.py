"""What the decode attention of one launch per projection reads, against what is live (host only)."""
import ctypes as C

import pytest

from homura_amd import _ffi


@pytest.mark.parametrize("max_len", [1, 64, 100, 128, 129, 1000, 2048, 3000, 8192, 32768])
def test_no_more_than_a_chunk_past_the_live_rows(max_len):
    """Splits that begin in rows that are surely live ask for their chunk unseen, so these rows have to be live at every length that the
    span serves, and the chunks that begin in them may reach past the live length by less than one of them, whatever the span covers."""
    lib, span, chunk, sure = _ffi.load(), C.c_int(), C.c_int(), C.c_int()
    for live in range(1, max_len + 1):
        assert lib.hm_test_attn_rows(live, max_len, C.byref(span), C.byref(chunk), C.byref(sure)) == 0
        assert live <= span.value <= max_len and 1 <= sure.value <= live, (live, span.value, sure.value)
        asked = min(-(-sure.value // chunk.value) * chunk.value, span.value)
        assert asked < live + chunk.value, (live, span.value, asked)
    assert lib.hm_test_attn_rows(max_len + 1, max_len, C.byref(span), C.byref(chunk), C.byref(sure)) != 0
