"""Tiles of the prompt pass's matrix products at the sizes where their choice turns (GPU)."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from homura_amd import DTYPE_F32, DTYPE_Q4_0, DTYPE_Q8_0, synth, synth_model
from homura_amd.runtime import HomuraError

pytestmark = pytest.mark.gpu


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


def test_prompt_longer_than_a_chunk(ctx):
    """4097 and 4400 tokens go through the layers in a chunk of 4096 and a rest. The rows they leave in the cache give the logits that
    the same tokens in portions of other sizes give, up to the cache rows that round to bf16 the other way (one ulp, 0.4 %,
    of single elements under softmax weights of 1 / 4000 a row)."""
    cfg = dataclasses.replace(synth_model.TINY, max_position_embeddings=4500)
    m = synth_model.build_model(ctx, cfg, synth_model.synth_weights(cfg, 5), 4500)
    for n in (4097, 4400):
        ids = synth.token_ids(n, n + 1, cfg.vocab_size)
        got = []
        for cuts in ((0, n), (0, 1111, 1700, n)):
            m.reset_kv_cache()
            for a, b in zip(cuts, cuts[1:]):
                m.prefill(ids[a:b], want_logits=False)
            assert m.kv_cache_len() == n
            got.append(m.run_kv(ids[n:])[0].astype(np.float64))
        assert np.abs(got[0] - got[1]).max() <= 2e-3 * np.abs(got[1]).max()
    m.reset_kv_cache()
    rows = m.prefill(ids[:1100])          # logits of more rows than are held at a time
    m.reset_kv_cache()
    m.prefill(ids[:600], want_logits=False)
    tail = m.prefill(ids[600:1100])
    assert np.abs(rows[600:] - tail).max() <= 2e-3 * np.abs(tail).max()
    m.close()


@pytest.mark.parametrize("M,K,N", [(130, 192, 264), (37, 448, 8), (200, 320, 136), (129, 256, 120), (65, 576, 392), (257, 704, 1032), (64, 1216, 72)])
def test_kn_products_between_whole_rounds(ctx, M, K, N):
    """[K, N] weights: none to three K tiles of 64 behind whole rounds of four, with and without a round ahead of them, columns
    that end inside a tile. Bound as above."""
    guard = 512
    a, b = synth.normal_bf16(61, M * K, 1.0).reshape(M, K), synth.normal_bf16(62, K * N, 0.02).reshape(K, N)
    da, db, dc = ctx.to_device(a), ctx.to_device(b), ctx.to_device(np.full(M * N + guard, -77.0, np.float32))
    ctx.gemm_bf16(da, db, dc, M, K, N)
    got = dc.download(np.float32, (M * N + guard,))
    assert np.all(got[M * N:] == -77.0), "wrote past the end of C"
    a64, b64 = synth.bf16_to_f32(a).astype(np.float64), synth.bf16_to_f32(b).astype(np.float64)
    assert np.all(np.abs(got[:M * N].reshape(M, N) - a64 @ b64) <= 3 * K * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64)))
    for buf in (da, db, dc):
        buf.free()


@pytest.mark.parametrize("groups", [None, 1, 2, 4])
@pytest.mark.parametrize("S,past,H,kvh,hd", [(640, 0, 12, 2, 128), (1000, 37, 16, 8, 128), (2111, 0, 14, 2, 64),
                                             (130, 65, 32, 4, 64), (4096, 0, 8, 8, 64), (4096, 0, 16, 8, 128), (4000, 0, 14, 2, 64)])
def test_prompt_attention_over_key_groups(ctx, monkeypatch, S, past, H, kvh, hd, groups):
    """The chosen number of key groups and each of them, heads in eighths and not, ragged row blocks, more than one round of
    workgroups with each. Keys and values are bf16, queries and
    probabilities carried whole, sums f32: 2^-20 of the largest value, over a few thousand additions, holds it."""
    monkeypatch.delenv("HOMURA_PREFILL_KEY_GROUPS", raising=False)
    if groups:
        monkeypatch.setenv("HOMURA_PREFILL_KEY_GROUPS", str(groups))
    rng = np.random.default_rng(S)
    L = past + S
    q = rng.standard_normal((S, H, hd)).astype(np.float32)
    k, v = (synth.f32_to_bf16_rne(rng.standard_normal((kvh, L, hd)).astype(np.float32)) for _ in range(2))
    dq, dk, dv, do = ctx.to_device(q), ctx.to_device(k), ctx.to_device(v), ctx.empty(S * H * hd)
    ctx.gqa_prefill_attn(dq, dk, dv, do, S, H, kvh, hd, L, past, hd ** -0.5)
    got = do.download(np.float32, (S, H, hd))
    k64, v64 = synth.bf16_to_f32(k).astype(np.float64), synth.bf16_to_f32(v).astype(np.float64)
    for i in (0, 1, 15, 16, 127, 128, S // 2, S - 2, S - 1):
        n = past + i + 1
        for h in range(0, H, max(1, H // 4)):
            g = h // (H // kvh)
            s = k64[g, :n] @ q[i, h].astype(np.float64) * hd ** -0.5
            p = np.exp(s - s.max())
            assert np.abs(got[i, h] - (p / p.sum()) @ v64[g, :n]).max() <= 2.0 ** -20 * 6
    for buf in (dq, dk, dv, do):
        buf.free()


@pytest.mark.parametrize("groups", [1, 2, 4])
@pytest.mark.parametrize("H,kvh,hd", [(16, 8, 128), (14, 2, 64)])
def test_prompt_rows_ahead_of_an_infinite_value(ctx, monkeypatch, groups, H, kvh, hd):
    """Rows of 16 that see none of the 32 keys around an infinite value stay finite, whatever a wavefront takes between barriers."""
    monkeypatch.setenv("HOMURA_PREFILL_KEY_GROUPS", str(groups))
    S = 300
    rng = np.random.default_rng(groups)
    q = rng.standard_normal((S, H, hd)).astype(np.float32)
    k, v = (synth.f32_to_bf16_rne(rng.standard_normal((kvh, S, hd)).astype(np.float32)) for _ in range(2))
    v[:, 190, 5] = 0x7F80
    dq, dk, dv, do = ctx.to_device(q), ctx.to_device(k), ctx.to_device(v), ctx.empty(S * H * hd)
    ctx.gqa_prefill_attn(dq, dk, dv, do, S, H, kvh, hd, S, 0, hd ** -0.5)
    got = do.download(np.float32, (S, H, hd))
    assert np.all(np.isfinite(got[:160])) and np.all(np.isfinite(np.delete(got, 5, 2))) and not np.any(np.isfinite(got[190:, :, 5]))
    for buf in (dq, dk, dv, do):
        buf.free()


@pytest.mark.parametrize("M,K,N", [(1, 32, 8), (7, 96, 200), (24, 1024, 6144), (31, 160, 4097), (32, 896, 33), (33, 32, 64), (37, 4864, 896),
                                   (64, 1056, 1001), (64, 1536, 17920), (64, 2080, 6150), (24, 96, 17920), (31, 96, 31501),
                                   (8, 2080, 200), (9, 1056, 97), (16, 544, 6150), (17, 1056, 1001), (25, 2080, 97), (48, 1056, 6150), (49, 544, 200)])
@pytest.mark.parametrize("form", ["f32", "bf16", "q8_0", "q4_0"])
def test_products_of_few_rows(ctx, oracle, form, M, K, N):
    """Row tiles of 32 and 64, one and two tiles of B, half a group of 64 k at the end, columns that end inside a vector, one
    round of workgroups and two, the last one full or not, rows on both sides of where a load of A more is made.
    Bound as above; the block formats' scales are one rounding more a block."""
    if form != "f32" and form != "bf16" and K % 64:
        K = (K + 63) // 64 * 64
    guard = 512
    x = synth.normal_f32(31, M * K).reshape(M, K)
    dc = ctx.to_device(np.full(M * N + guard, -77.0, np.float32))
    if form in ("q8_0", "q4_0"):
        raw = {"q8_0": synth.q8_0_blocks, "q4_0": synth.q4_0_blocks}[form](41, N * K // 32, 0.01)
        w64 = getattr(oracle, "dequant_" + form)(raw).reshape(N, K).astype(np.float64)
        dx, dw = ctx.to_device(x), ctx.to_device(raw)
        ctx.gemm_f32_quant_nk(dx, dw, {"q8_0": DTYPE_Q8_0, "q4_0": DTYPE_Q4_0}[form], dc, M, K, N)
    else:
        w = synth.normal_bf16(32, K * N, 0.02).reshape(N, K)
        w64 = synth.bf16_to_f32(w).astype(np.float64)
        if form == "bf16":
            bits = synth.f32_to_bf16_rne(x)
            x = synth.bf16_to_f32(bits)
            dx, dw = ctx.to_device(bits), ctx.to_device(w)
            ctx.gemm_bf16_nk(dx, dw, dc, M, K, N)
        else:
            dx, dw = ctx.to_device(x), ctx.to_device(w)
            ctx.gemm_f32_bf16_nk(dx, dw, dc, M, K, N)
    got = dc.download(np.float32, (M * N + guard,))
    assert np.all(got[M * N:] == -77.0), "wrote past the end of C"
    x64 = x.astype(np.float64)
    bound = 4 * K * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64).T)
    assert np.all(np.abs(got[:M * N].reshape(M, N) - x64 @ w64.T) <= bound)
    for buf in (dx, dw, dc):
        buf.free()


@pytest.mark.parametrize("K,N", [(32, 1), (32, 2801), (992, 5603), (1024, 11203), (1024, 45001), (1056, 1401), (2048, 22403), (2080, 703),
                                 (4096, 11201), (4128, 701), (7680, 5601), (64, 3999), (480, 4003), (512, 20001), (1152, 60000), (1536, 60001),
                                 (2432, 16500), (2432, 10241), (2496, 10241), (2560, 10240), (2560, 16501), (3264, 60000), (3584, 60001), (4128, 15003), (4352, 14999), (4384, 15000), (5120, 15001),
                                 (7712, 1001), (8192, 5601), (8192, 8003)])
def test_q8_0_rows_straight_from_blocks(ctx, oracle, K, N):
    """Half a, one, two and four wavefronts a row, one, two and five chunks each, every number of rows a set, rows and units past the
    end; the sizes from which rows go through LDS; rows that no LDS stage holds, and a matrix whose planes no workspace would.
    A block's sum is 32 f32 additions of exact integers times activations, the blocks' sums as many again as there are."""
    raw = synth.q8_0_blocks(51, N * K // 32, 0.01)
    x = synth.normal_f32(52, 2 * K).reshape(2, K)
    dx, dw, dout = ctx.to_device(x), ctx.to_device(raw), ctx.to_device(np.full(2 * N + 64, -77.0, np.float32))
    ctx.gemv_q8_0(dx, dw, dout, 2, K, N)
    got = dout.download(np.float32, (2 * N + 64,))
    assert np.all(got[2 * N:] == -77.0), "wrote past the end"
    w64, x64 = oracle.dequant_q8_0(raw).reshape(N, K).astype(np.float64), x.astype(np.float64)
    blocks = raw.reshape(-1, 34)
    scale = np.abs(blocks[:, :2].copy().view(np.float16).astype(np.float64)).reshape(N, K // 32)
    # quants enter as q + 128 and the offset is taken off a block: magnitudes of up to 256 scales
    mags = np.abs(x64).reshape(2, K // 32, 32).sum(2) @ (256 * scale).T
    assert np.all(np.abs(got[:2 * N].reshape(2, N) - x64 @ w64.T) <= (64 + K / 16) * 2.0 ** -24 * mags)
    for buf in (dx, dw, dout):
        buf.free()


@pytest.mark.parametrize("K", [32, 544, 1056, 2080, 4128])
def test_q8_0_row_with_an_infinite_scale(ctx, K):
    """A first block with an infinite scale and positive products makes its row infinite, also where the row's last units are
    past its end; the other rows are what they are without it."""
    N = 5
    raw = synth.q8_0_blocks(51, N * K // 32, 0.01).reshape(N, K // 32, 34).copy()
    x = np.abs(synth.normal_f32(52, K)) + np.float32(0.1)
    dx, dout = ctx.to_device(x), ctx.empty(N)
    got = []
    for inf in (False, True):
        if inf:
            raw[2, 0, :2], raw[2, 0, 2:] = (0x00, 0x7C), 3
        dw = ctx.to_device(raw)
        ctx.gemv_q8_0(dx, dw, dout, 1, K, N)
        got.append(dout.download(np.float32, (N,)))
        dw.free()
    assert got[1][2] == np.inf and np.array_equal(np.delete(got[0], 2), np.delete(got[1], 2))
    for buf in (dx, dout):
        buf.free()


# one, two and four wavefronts a row, one chunk to three, units past the row's end in the last one (Q4_0: rows that are cut at all)
@pytest.mark.parametrize("block", [0, -1])
@pytest.mark.parametrize("fmt,K", [("q8_0", k) for k in (544, 1056, 2080, 4128, 6176, 8960)] + [("q4_0", k) for k in (4128, 6176, 8960)])
def test_planes_row_with_an_infinite_scale(ctx, fmt, K, block):
    """As above from planes, the infinite scale in the first block or in the last."""
    N, size = 5, 34 if fmt == "q8_0" else 18
    raw = (synth.q8_0_blocks if fmt == "q8_0" else synth.q4_0_blocks)(51, N * K // 32, 0.01).reshape(N, K // 32, size).copy()
    x = np.abs(synth.normal_f32(52, K)) + np.float32(0.1)
    dx, dout = ctx.to_device(x), ctx.empty(N)
    got = []
    for inf in (False, True):
        if inf:
            raw[2, block, :2], raw[2, block, 2:] = (0x00, 0x7C), 3 if fmt == "q8_0" else 0xCC
        dw = ctx.to_device(raw)
        planes = ctx.pack_quant_planes(DTYPE_Q8_0 if fmt == "q8_0" else DTYPE_Q4_0, dw, N, K)
        (ctx.gemv_q8_0_planes if fmt == "q8_0" else ctx.gemv_q4_0_planes)(dx, planes, dout, 1, K, N)
        got.append(dout.download(np.float32, (N,)))
        dw.free()
        planes.free()
    assert got[1][2] == np.inf and np.array_equal(np.delete(got[0], 2), np.delete(got[1], 2))
    for buf in (dx, dout):
        buf.free()


@pytest.mark.parametrize("n", [127, 255, 256, 300, 1025, 2048])
def test_selective_scan_in_segments(ctx, n):
    """A chunk scanned in segments leaves the logits that the same tokens give one portion of at most 100 after the other
    (those are one segment each), on an empty state and behind one."""
    cfg = {"architecture": "Nokuvik", "vocab": 96, "width": 64, "embedding": {"scale": 1.0}, "norm": {"eps": 1e-5}, "loop": None,
           "layers": [{"type": "mamba1", "mlp": None, "mixer": {"inner": 128, "conv": 4, "dt_rank": 8, "state": s}} for s in (16, 24, 40, 100)]}
    m = synth_model.build_block_model(ctx, cfg, 3, 4096, DTYPE_F32)
    ids = synth.token_ids(n, n + 51, cfg["vocab"])
    for past in (0, 50):
        got = []
        for step in (n, 100):
            m.reset_kv_cache()
            if past:
                m.prefill(ids[:past], want_logits=False)
            out = [m.prefill(ids[at:min(at + step, past + n)]) for at in range(past, past + n, step)]
            got.append((np.concatenate(out).astype(np.float64), m.run_kv(ids[past + n:past + n + 1])[0].astype(np.float64)))
        for a, b in zip(*got):
            assert np.abs(a - b).max() <= 2e-4 * np.abs(b).max()
    m.close()


# one chunk at its limit, two of uneven and of equal rows, five
@pytest.mark.parametrize("n", [512, 513, 1024, 2050])
def test_gated_recurrence_in_chunks(ctx, n):
    """As above for rows that one workgroup does not hold: chunks of them against portions of 100, the tolerance as there. Widths on
    both sides of a workgroup's 16 channels, filter histories that reach across the portions."""
    cfg = {"architecture": "Nokuvik", "vocab": 96, "width": 64, "embedding": {"scale": 1.0}, "norm": {"eps": 1e-5}, "loop": None,
           "layers": [{"type": "rglru", "mlp": None, "mixer": {"width": w, "conv": c, "blocks": b}} for w, c, b in ((60, 3, 3), (64, 4, 1), (144, 2, 9))]}
    m = synth_model.build_block_model(ctx, cfg, 3, 4096, DTYPE_F32)
    ids = synth.token_ids(n, n + 51, cfg["vocab"])
    for past in (0, 50):
        got = []
        for step in (n, 100):
            m.reset_kv_cache()
            if past:
                m.prefill(ids[:past], want_logits=False)
            out = [m.prefill(ids[at:min(at + step, past + n)]) for at in range(past, past + n, step)]
            got.append((np.concatenate(out).astype(np.float64), m.run_kv(ids[past + n:past + n + 1])[0].astype(np.float64)))
        for a, b in zip(*got):
            assert np.abs(a - b).max() <= 2e-4 * np.abs(b).max()
    m.close()


# whole chunks of 512 rows, with a last one of 88 and of 300 rows; of 8192 channels a pair of launches takes four chunks
@pytest.mark.parametrize("n,shapes", [(n, ((60, 3, 3), (64, 4, 1), (144, 2, 9))) for n in (1024, 1112, 2348, 4096)] + [(2348, ((8192, 4, 128),))])
def test_gated_recurrence_in_one_pass_as_in_portions(ctx, n, shapes):
    """A prompt of several chunks in one pass against portions of a chunk each, whose states go through memory: the same bits, for the
    products of these widths add up alike whatever the rows (one slice, 32-bit sums in order)."""
    cfg = {"architecture": "Nokuvik", "vocab": 96, "width": 64, "embedding": {"scale": 1.0}, "norm": {"eps": 1e-5}, "loop": None,
           "layers": [{"type": "rglru", "mlp": None, "mixer": {"width": w, "conv": c, "blocks": b}} for w, c, b in shapes]}
    m = synth_model.build_block_model(ctx, cfg, 3, 8192, DTYPE_F32)
    ids = synth.token_ids(n + 1, n + 1, cfg["vocab"])
    got = []
    for step in (n, 512):
        m.reset_kv_cache()
        rows = [m.prefill(ids[at:min(at + step, n)]) for at in range(0, n, step)]
        got.append((np.concatenate(rows), m.run_kv(ids[n:n + 1])))
    for a, b in zip(*got):
        assert np.array_equal(a, b)
    m.close()


def test_long_k_quant_prompt_with_wide_rows(ctx):
    """Rows of 18 blocks need two K slices (a workgroup's tables hold 16), also where the tiles alone fill the chip."""
    cfg = synth_model.TransformerConfig(hidden_size=2048, intermediate_size=4608, num_attention_heads=16, num_hidden_layers=1, vocab_size=512,
                                        num_key_value_heads=4, head_dim=64, max_position_embeddings=2048, tie_word_embeddings=False)
    types = synth_model.q4_k_m_mix(cfg)
    m = synth_model.build_model(ctx, cfg, synth_model.synth_weights(cfg, 9, DTYPE_Q8_0, False, proj_dtypes=types), 2048, DTYPE_Q8_0, False,
                                proj_dtypes=types)
    ids = synth.token_ids(6, 1501, cfg.vocab_size)
    got = []
    for cuts in ((0, 1500), (0, 400, 800, 1200, 1500)):
        m.reset_kv_cache()
        for a, b in zip(cuts, cuts[1:]):
            m.prefill(ids[a:b], want_logits=False)
        got.append(m.run_kv(ids[1500:])[0].astype(np.float64))
    # one layer: the sums are integers, only rows whose norm rounds the other way are quantised differently (1 / 127 of a value)
    assert np.abs(got[0] - got[1]).max() <= 1e-2 * np.abs(got[1]).max()
    m.close()


@pytest.mark.parametrize("fmt", [DTYPE_Q8_0, DTYPE_Q4_0])
def test_long_block_format_prompt_of_a_narrow_model(ctx, fmt):
    """A width below a K-quant block and a wide MLP: 1100 rows of 8192 gate and up values are more than the least that a product's
    scratch holds. The same tokens in short portions leave the same rows, up to cache elements that round the other way."""
    cfg = synth_model.TransformerConfig(hidden_size=128, intermediate_size=4096, num_attention_heads=2, num_hidden_layers=2, vocab_size=256,
                                        num_key_value_heads=1, head_dim=64, max_position_embeddings=1200, tie_word_embeddings=False)
    types = [fmt] * 7 * cfg.num_hidden_layers
    m = synth_model.build_model(ctx, cfg, synth_model.synth_weights(cfg, 11, DTYPE_Q8_0, False, proj_dtypes=types), 1200, DTYPE_Q8_0, False,
                                proj_dtypes=types)
    ids = synth.token_ids(7, 1101, cfg.vocab_size)
    got = []
    for step in (1100, 100):
        m.reset_kv_cache()
        rows = [m.prefill(ids[at:at + step]) for at in range(0, 1100, step)]
        got.append((np.concatenate(rows).astype(np.float64), m.run_kv(ids[1100:])[0].astype(np.float64)))
    for a, b in zip(*got):
        assert np.abs(a - b).max() <= 2e-3 * np.abs(b).max()
    m.close()


@pytest.mark.parametrize("B,H,kvh,hd,kv_len", [(1, 7, 1, 64, 65), (1, 4, 2, 128, 513), (2, 12, 2, 128, 1025), (1, 8, 1, 64, 2047), (3, 32, 4, 64, 577)])
def test_fold_of_a_few_splits(ctx, B, H, kvh, hd, kv_len):
    """Two to thirty-two splits, one far ahead of the others: the weights of the fold span the whole range of exp."""
    rng = np.random.default_rng(kv_len)
    q = rng.standard_normal((B, H, hd)).astype(np.float32)
    k, v = rng.standard_normal((2, B, kvh, kv_len, hd)).astype(np.float32)
    k[:, :, kv_len // 2] *= 20.0
    kb, vb = synth.f32_to_bf16_rne(k), synth.f32_to_bf16_rne(v)
    dq, dk, dv, do = ctx.to_device(q), ctx.to_device(kb), ctx.to_device(vb), ctx.empty(B * H * hd)
    ctx.gqa_decode_attn(dq, dk, dv, do, B, H, kvh, hd, kv_len, kv_len, hd ** -0.5)
    got = do.download(np.float32, (B, H, hd))
    k64, v64 = synth.bf16_to_f32(kb).astype(np.float64), synth.bf16_to_f32(vb).astype(np.float64)
    for b in range(B):
        for h in range(H):
            s = k64[b, h // (H // kvh)] @ q[b, h].astype(np.float64) * hd ** -0.5
            p = np.exp(s - s.max())
            # scores up to about 60 in f32: an exponential is off by 2^-24 of its exponent
            assert np.abs(got[b, h] - (p / p.sum()) @ v64[b, h // (H // kvh)]).max() <= 5e-5
    for buf in (dq, dk, dv, do):
        buf.free()


@pytest.mark.parametrize("H,kvh,hd,kv_len", [(8, 2, 128, 577), (4, 2, 64, 300), (12, 2, 128, 200), (32, 4, 64, 2047)])
def test_fold_keeps_an_infinite_value(ctx, H, kvh, hd, kv_len):
    """An infinite element of the last split's values makes its own column infinite, however many splits there are, and no other."""
    rng = np.random.default_rng(kv_len)
    q = rng.standard_normal((1, H, hd)).astype(np.float32)
    k, v = (synth.f32_to_bf16_rne(rng.standard_normal((1, kvh, kv_len, hd)).astype(np.float32)) for _ in range(2))
    v[:, :, kv_len - 1, 5] = 0x7F80
    dq, dk, dv, do = ctx.to_device(q), ctx.to_device(k), ctx.to_device(v), ctx.empty(H * hd)
    ctx.gqa_decode_attn(dq, dk, dv, do, 1, H, kvh, hd, kv_len, kv_len, hd ** -0.5)
    got = do.download(np.float32, (H, hd))
    assert np.all(got[:, 5] == np.inf) and np.all(np.isfinite(np.delete(got, 5, 1)))
    for buf in (dq, dk, dv, do):
        buf.free()


def die_folds(c):
    n = (C.c_longlong * 3)()
    c._check(c.lib.hm_test_routes(c.h, n))
    return n[0]


# the kernel that holds its chunk in registers, and the one that walks it
@pytest.mark.parametrize("B,H,kvh,hd,kv_len", [(1, 16, 8, 128, 1000), (8, 12, 2, 128, 4096)])
def test_splits_from_several_dies_are_not_folded_silently(ctx, B, H, kvh, hd, kv_len):
    """Arrivals from two dies in a group that is dealt to one: the launch ends as ever, the synchronisations behind it fail and go on failing,
    and another context takes no harm."""
    c = type(ctx)(0)
    dq, dk, dv, do = c.to_device(np.ones((B, H, hd), np.float32)), *(c.to_device(np.zeros((B, kvh, kv_len, hd), np.uint16)) for _ in range(2)), c.empty(B * H * hd)
    call = lambda: c.gqa_decode_attn(dq, dk, dv, do, B, H, kvh, hd, kv_len, kv_len, hd ** -0.5)
    before = die_folds(c)
    call()
    assert die_folds(c) == before + 1
    assert np.all(do.download(np.float32) == 0)
    c._check(c.lib.hm_test_die_arrivals(c.h, 3))
    call()
    for _ in range(2):
        with pytest.raises(HomuraError, match="HOMURA_FOLD_LAUNCH"):
            c.sync()
        with pytest.raises(HomuraError, match="HOMURA_FOLD_LAUNCH"):
            do.download(np.float32)
    for buf in (dq, dk, dv, do):
        buf.free()
    c.close()
    ctx.sync()


# Groups of splits that sit on one die each: one to eight heads of a workgroup (four, two or one share of the splits a thread), two to
# thirty-two splits, four groups and as many as the dies hold, both kernels; and the same through a fold in a launch of its own
@pytest.mark.parametrize("B,H,kvh,hd,kv_len", [(4, 1, 1, 64, 65), (1, 32, 32, 64, 500), (4, 4, 1, 128, 600), (8, 3, 1, 128, 2047), (1, 16, 8, 128, 1000),
                                               (8, 12, 2, 128, 4096), (8, 14, 2, 64, 5000), (4, 64, 8, 128, 4001), (16, 5, 1, 64, 4096),
                                               (6, 14, 2, 64, 777)])
def test_splits_folded_on_their_die(ctx, monkeypatch, B, H, kvh, hd, kv_len):
    """Eager twice and replayed three times (the arrivals are counted anew every time), with other work between, in a context that folds so and in
    one that does not. A softmax over f32 sums:
    2^-20 of the largest value holds a few thousand additions, and the long caches' two-piece operands 2^-17 of their terms."""
    rng = np.random.default_rng(kv_len + H)
    q = rng.standard_normal((B, H, hd)).astype(np.float32)
    k, v = (synth.f32_to_bf16_rne(rng.standard_normal((B, kvh, kv_len, hd)).astype(np.float32)) for _ in range(2))
    k64, v64 = (np.repeat(synth.bf16_to_f32(x).astype(np.float64), H // kvh, 1) for x in (k, v))
    s = np.einsum("bhnd,bhd->bhn", k64, q.astype(np.float64)) * hd ** -0.5
    p = np.exp(s - s.max(-1, keepdims=True))
    want = np.einsum("bhn,bhnd->bhd", p / p.sum(-1, keepdims=True), v64)
    monkeypatch.setenv("HOMURA_FOLD_LAUNCH", "1")
    apart = type(ctx)(0)
    got = []
    for c in (ctx, apart):
        dq, dk, dv, do, other = c.to_device(q), c.to_device(k), c.to_device(v), c.empty(B * H * hd), c.empty(256 * hd)
        call = lambda out: c.gqa_decode_attn(dq, dk, dv, out, B, H, kvh, hd, kv_len, kv_len, hd ** -0.5)
        before = die_folds(c)
        for _ in range(2):
            call(do)
        assert die_folds(c) - before == (2 if c is ctx else 0)
        got.append(do.download(np.float32, (B, H, hd)))
        graph = C.c_void_p()
        c._check(c.lib.hm_graph_begin(c.h))
        call(do)
        c.gqa_decode_attn(dq, dk, dv, other, 1, H // kvh, 1, hd, kv_len, min(kv_len, 300), hd ** -0.5)
        c._check(c.lib.hm_graph_end(c.h, C.byref(graph)))
        for _ in range(3):
            c._check(c.lib.hm_fill_zero(c.h, do.ptr, B * H * hd * 4))
            c._check(c.lib.hm_graph_launch(c.h, graph, 1))
            assert np.array_equal(do.download(np.float32, (B, H, hd)), got[-1])
            c.gqa_decode_attn(dq, dk, dv, other, 1, H // kvh, 1, hd, kv_len, kv_len, hd ** -0.5)
        c._check(c.lib.hm_graph_destroy(c.h, graph))
        for buf in (dq, dk, dv, do, other):
            buf.free()
    apart.close()
    for out in got:
        assert np.abs(out - want).max() <= 2.0 ** -17 * np.abs(v64).max()
    assert np.abs(got[0] - got[1]).max() <= 2.0 ** -21 * np.abs(v64).max()
