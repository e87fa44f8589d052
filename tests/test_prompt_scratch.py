"""What the prompt pass sets aside for its products, against what the products write (host only)."""
import ctypes as C

import numpy as np
import pytest

from homura_amd import DTYPE_BF16, DTYPE_Q4_0, DTYPE_Q4_K, DTYPE_Q6_K, DTYPE_Q8_0, _ffi
from test_gpu_product_tiles import TILES

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


@pytest.mark.parametrize("kind", [0, 1, 2])
def test_every_tile_of_the_products_is_tested(kind):
    """The products that the GPU tests name by their tile get that tile, and 20000 products spread over the sizes of prompts and
    models get no tile that is not among them: a new fit of the timings that moves one of them shows here."""
    lib, tm, tn, slices = _ffi.load(), C.c_int(), C.c_int(), C.c_int()

    def pick(m, k, n):
        assert lib.hm_test_product_tiles(kind, m, k, n, 256, 8, C.byref(tm), C.byref(tn), C.byref(slices)) == 0
        return tm.value, tn.value, slices.value > 1
    named = {tile: shape for kd, tile, shape in TILES if kd == kind}
    for tile, shape in named.items():
        assert pick(*shape) == tile and shape[0] % tile[0] and shape[2] % tile[1]
    rng = np.random.default_rng(kind)
    for m, k, n in zip(2 ** rng.uniform(0, 12.01, 20000), 2 ** rng.uniform(0, 7.2, 20000), 2 ** rng.uniform(3, 15, 20000)):
        assert pick(int(m), 64 * int(k), int(n)) in named, (int(m), 64 * int(k), int(n))
