"""Tiles of the prompt pass's matrix products at the sizes where their choice turns (GPU)."""
import numpy as np
import pytest

from homura_amd import Context, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with Context(0) as c:
        yield c


@pytest.mark.parametrize("M,K,N", [(1100, 32, 4000), (1100, 96, 4000), (1025, 1024, 4001), (2048, 256, 4096), (1153, 64, 3841)])
def test_wide_tiles_of_the_piece_product(ctx, M, K, N):
    """More 128 x 128 tiles than CUs: 128 x 256 tiles, whole and ragged, an even and an odd number of 32-deep stages.
    Products of bf16 x bf16 are exact and every sum is f32: K additions of at most 2^-24 of the running sum each, which
    stays below the sum of magnitudes."""
    x = synth.normal_f32(21, M * K).reshape(M, K)
    w = synth.normal_bf16(22, K * N, 0.02).reshape(N, K)
    guard = 1024
    dx, dw, dc = ctx.to_device(x), ctx.to_device(w), ctx.to_device(np.full(M * N + guard, -77.0, np.float32))
    ctx.gemm_f32_bf16_nk(dx, dw, dc, M, K, N)
    got = dc.download(np.float32, (M * N + guard,))
    assert np.all(got[M * N:] == -77.0), "wrote past the end of C"
    x64, w64 = x.astype(np.float64), synth.bf16_to_f32(w).astype(np.float64)
    bound = 3 * K * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64).T)
    assert np.all(np.abs(got[:M * N].reshape(M, N) - x64 @ w64.T) <= bound)
    for buf in (dx, dw, dc):
        buf.free()
