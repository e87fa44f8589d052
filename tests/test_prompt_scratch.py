"""What the prompt pass sets aside for its products, against what the products write (host only)."""
import ctypes as C

import pytest

from homura_amd import DTYPE_BF16, DTYPE_Q4_0, DTYPE_Q4_K, DTYPE_Q6_K, DTYPE_Q8_0, _ffi

ROWS = [1, 8, 32, 33, 64, 65, 128, 500, 1025, 2048, 3000, 4096]


@pytest.mark.parametrize("dtype", [DTYPE_BF16, DTYPE_Q8_0, DTYPE_Q4_0, DTYPE_Q4_K, DTYPE_Q6_K])
@pytest.mark.parametrize("K", [64, 128, 192, 256, 896, 1024, 4096, 4608, 8960, 32768])
def test_prompt_products_fit_their_scratch(dtype, K):
    lib = _ffi.load()
    held, written = C.c_longlong(), C.c_longlong()
    for cus in (64, 256):
        for N in (128, 384, 1024, 4096, 8192, 28672):
            for m in ROWS:
                for rows in (r for r in (128, 256, 512, 1024, 2048, 4096) if r >= m):
                    assert lib.hm_test_prompt_product(dtype, rows, m, K, N, cus, C.byref(held), C.byref(written)) == 0
                    assert written.value <= held.value, (cus, N, m, rows)
