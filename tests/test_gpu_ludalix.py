"""Ludalix models on the GPU against the numpy oracle: every mechanism alone, prompts in one piece and in portions,
decoding, windows, kept tokens and their edges, shared caches, extreme gates, reuse of the cache, generation. `f32` runs
everything in 32 bits; `bf16` is the serving precision."""
from __future__ import annotations

import json

import numpy as np
import pytest

import homura_amd
import ludalix_fixture as lf
import ludalix_oracle as lo
from homura_amd import trace
from homura_amd.runtime import DTYPE_BF16, DTYPE_F32, HomuraError, Rng, SamplingConfig, sample_token_host
from test_gpu_block_model import feed, tokens, write_model

pytestmark = pytest.mark.gpu

DTYPES = {"f32": DTYPE_F32, "bf16": DTYPE_BF16}
# worst row, and the limit for all but one row in fifty: where a normaliser of a matrix memory comes out near zero, its row
# magnifies every rounding ahead of it
LIMIT = {"f32": 3e-4, "bf16": 1.0}
MOST = {"f32": 2e-5, "bf16": 0.04}


def say(msg):
    print(f"[ludalix] {msg}", flush=True)


def verdict(got, want, dtype, what=""):
    rows = np.array([lf.error(got[i:i + 1], want[i:i + 1]) * want[i].std() / want.std() for i in range(len(want))])
    most = np.sort(rows)[-1 - len(rows) // 50]
    say(f"{what} worst {rows.max():.2e} at {rows.argmax()}, most {most:.2e}")
    assert rows.max() < LIMIT[dtype] and most < MOST[dtype], (what, dtype)


def run(ctx, cfg, w, toks, want, dtype, cuts=(), prefill_min=8, max_len=None, chunk=None):
    m = lf.build(ctx, cfg, w, max_len or len(toks), DTYPES[dtype], chunk)
    m.set_prefill_min(prefill_min)
    got = feed(m, toks, cuts)
    m.close()
    verdict(got, want, dtype, f"{len(toks)} tokens, {dtype}, cuts {list(cuts)[:6]}, prefill_min {prefill_min}, chunk {chunk}:")
    return got


def check(ctx, cfg, n, dtype, seed=0, gates=(0.0, 2.0), **kw):
    say(json.dumps(cfg["layers"])[:200])
    seeds = range(seed, seed + (1 if dtype == "f32" or not any(l["mlp"] and l["mlp"]["kind"] == "moe" for l in cfg["layers"]) else 12))
    _, w, toks, want, _ = lf.clearest(cfg, n, seeds, gates)
    run(ctx, cfg, w, toks, want, dtype, **kw)


# ── each mechanism alone, in a prompt and token by token ──

ONE_LAYER = {
    "attention": lf.attn(),
    "attention_no_mask": lf.attn(window=None),
    "attention_nothing_kept": lf.attn(keep=0),
    "attention_window_1": lf.attn(window=1, keep=0),
    "attention_window_1_one_kept": lf.attn(window=1, keep=1),
    "attention_more_kept_than_window": lf.attn(window=4, keep=40),
    "attention_one_head": lf.attn(heads=1, kv_heads=1, dim=3, vdim=1),
    "attention_own_keys": lf.attn(heads=5, kv_heads=5),
    "attention_one_key_head": lf.attn(heads=7, kv_heads=1, dim=9, vdim=11),
    "attention_full_width": lf.attn(heads=4, kv_heads=2, dim=64, vdim=64),
    "attention_wide_keys": lf.attn(heads=4, kv_heads=2, dim=100, vdim=30),
    "attention_wide_values": lf.attn(heads=3, kv_heads=3, dim=10, vdim=128),
    "attention_widest": lf.attn(heads=2, kv_heads=1, dim=256, vdim=250),
    "memory": lf.memory(),
    "memory_one_head": lf.memory(heads=1, dim=1, vdim=1),
    "memory_tile_exactly": lf.memory(heads=2, dim=64, vdim=16),
    "memory_tile_less_one": lf.memory(heads=2, dim=63, vdim=15),
    "memory_many_heads": lf.memory(heads=19, dim=5, vdim=3),
    "memory_values_narrow": lf.memory(heads=2, dim=65, vdim=4),
    "memory_128": lf.memory(heads=2, dim=128, vdim=40),
    "memory_200": lf.memory(heads=2, dim=200, vdim=33),
    "memory_256": lf.memory(heads=1, dim=256, vdim=64),
    "memory_wide": lf.memory(heads=1, dim=300, vdim=18),
    "memory_512": lf.memory(heads=2, dim=512, vdim=100),
    "memory_widest": lf.memory(heads=1, dim=1000, vdim=20),
    "memory_values_wide": lf.memory(heads=1, dim=12, vdim=1100),
    "memory_small_cap": lf.memory(cap=0.3),
    "dense": lf.memory(heads=1, dim=2, vdim=2, mlp=lf.dense(ff=96)),
    "dense_tight": lf.attn(mlp=lf.dense(ff=37, limit=0.2)),
    "experts": lf.attn(mlp=lf.moe()),
    "experts_one": lf.attn(mlp=lf.moe(experts=1, top=1)),
    "experts_all": lf.attn(mlp=lf.moe(experts=4, top=4, ff=32)),
    "experts_many_places": lf.attn(mlp=lf.moe(experts=12, top=11, ff=9)),
    "experts_many": lf.attn(mlp=lf.moe(experts=70, top=3, ff=5)),
    "experts_very_many": lf.attn(mlp=lf.moe(experts=300, top=2, ff=3)),
    "experts_wide": lf.attn(mlp=lf.moe(experts=3, top=2, ff=1200)),
}


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("name", list(ONE_LAYER))
def test_one_mechanism(ctx, name, dtype):
    if name in ("attention_one_head", "memory_one_head") and dtype == "bf16":
        pytest.skip("a norm over one to three values takes their bf16 rounding to any size")
    cfg = lf.config([ONE_LAYER[name]])
    check(ctx, cfg, 140, dtype)
    check(ctx, cfg, 45, dtype, seed=20, prefill_min=0)


# heads that the output projection takes as they come: of 8 to 64 lanes, fewer than a wavefront's, the longest row; and the next beyond
# each limit
@pytest.mark.parametrize("heads,vdim", [(1, 64), (9, 64), (3, 128), (4, 256), (8, 256), (9, 256), (1, 512), (4, 512), (5, 512), (8, 512), (9, 512),
                                        (3, 32), (2, 96), (1, 1024)])
def test_memory_heads_in_the_output_projection(ctx, heads, vdim):
    check(ctx, lf.config([lf.memory(heads=heads, dim=24, vdim=vdim), lf.memory(heads=heads, dim=24, vdim=vdim)]), 24, "f32", prefill_min=0)


@pytest.mark.parametrize("width", [4096, 4160])  # the most outputs that take the heads as they come, and the next
def test_memory_heads_of_a_wide_model(ctx, width):
    check(ctx, lf.config([lf.memory(heads=3, dim=24, vdim=64)], width=width), 8, "f32", prefill_min=0)


# rows that end inside a wavefront, at one, and at a workgroup's last
@pytest.mark.parametrize("heads,vdim", [(3, 64), (4, 256), (3, 512), (4, 512)])
def test_memory_heads_without_an_eps(ctx, heads, vdim):
    check(ctx, lf.config([lf.memory(heads=heads, dim=24, vdim=vdim)], eps=0.0), 12, "f32", prefill_min=0)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("width,ff,experts,top", [(64, 64, 3, 1), (128, 200, 6, 2), (320, 128, 2, 2), (192, 448, 40, 5)])
def test_expert_products(ctx, width, ff, experts, top, dtype):
    """Row tiles of a group: none, ragged ones, several; products of one K tile and of many."""
    cfg = lf.config([lf.memory(heads=1, dim=4, vdim=12, mlp=lf.moe(experts=experts, top=top, ff=ff))], width=width)
    check(ctx, cfg, 700, dtype)
    check(ctx, cfg, 30, dtype, seed=40, cuts=range(12, 30))


# the router in the experts' launch: up to 36 and 64 of them, rows of up to 1024 and 2048, the largest router and one past it, rows that end
# inside a wavefront's load, as many places as experts, more pairs of rows than the launch has wavefronts
@pytest.mark.parametrize("width,experts,top,ff", [(1024, 36, 4, 40), (1056, 37, 3, 33), (1024, 64, 64, 32), (1056, 62, 2, 64), (1056, 63, 2, 64), (2048, 32, 2, 64), (2080, 9, 2, 40),
                                                  (200, 65, 5, 64), (300, 8, 4, 900)])
def test_router_in_the_experts_launch(ctx, width, experts, top, ff):
    cfg = lf.config([lf.memory(heads=1, dim=4, vdim=12, mlp=lf.moe(experts=experts, top=top, ff=ff)), lf.attn(mlp=lf.moe(experts=experts, top=top, ff=ff))],
                    width=width)
    check(ctx, cfg, 12, "f32", prefill_min=0)


@pytest.mark.parametrize("gates", [(-6.0, 3.0), (5.0, -4.0), (-6.0, -6.0), (6.0, 6.0)])
def test_extreme_gates(ctx, gates):
    """Input gates far below the running maximum's start and above it, memories that are forgotten at once or never."""
    cfg = lf.config([lf.memory(cap=12.0), lf.memory(heads=1, dim=70, vdim=30, cap=12.0)])
    check(ctx, cfg, 300, "f32", gates=gates, cuts=[130, 131, 132, 133, 290])
    check(ctx, cfg, 80, "f32", gates=gates, prefill_min=0)


MIXED = [lf.memory(mlp=lf.dense()), lf.attn(mlp=lf.moe(), keep=5), lf.memory(heads=2, dim=33, vdim=20, mlp=lf.moe(experts=4, top=1)),
         lf.attn(kv_from=1, keep=2, window=11, scale=0.3), lf.attn(heads=4, kv_heads=4, window=40, keep=1, mlp=lf.dense(ff=31, limit=0.5)),
         lf.attn(kv_from=1, heads=2, keep=9, window=33, mlp=lf.moe(experts=3, top=2))]


@pytest.mark.parametrize("width", [33, 40, 96, 260, 1100])
def test_other_widths(ctx, width):
    cfg = lf.config(MIXED, width=width, vocab=517, eps=1e-6, mult=1.0, scale=3.0)
    check(ctx, cfg, 40, "f32", seed=3)
    check(ctx, cfg, 20, "f32", seed=3, prefill_min=0)


def test_residual_behind_every_layer(ctx):
    cfg = lf.config(MIXED)
    _, w, toks, _, trail = lf.clearest(cfg, 50, [5])
    m = lf.build(ctx, cfg, w, 64, DTYPE_F32)
    m.capture_residuals()
    m.prefill(toks)
    got = m.captured_residuals(len(trail), len(toks))
    m.close()
    for i, (g, t) in enumerate(zip(got, trail)):
        assert lf.error(g, t) < 1e-5, f"layer {i}"


# ── portions ──

@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("size", [2, 3, 7, 8, 9, 31, 64])
def test_portions(ctx, size, dtype):
    check(ctx, lf.config(MIXED), 150, dtype, cuts=range(size, 150, size))


def test_portions_of_changing_size_then_single_tokens(ctx):
    cuts = list(np.cumsum([1, 40, 2, 8, 3, 17, 5, 9, 2, 2, 30])) + list(range(120, 150))
    check(ctx, lf.config(MIXED), 150, "f32", cuts=cuts)
    check(ctx, lf.config(MIXED), 150, "bf16", cuts=cuts)


@pytest.mark.parametrize("chunk", [16, 33, 64, 100])
def test_small_chunks_and_a_ring_that_goes_round(ctx, chunk):
    cfg = lf.config(MIXED)
    check(ctx, cfg, 330, "f32", chunk=chunk)
    check(ctx, cfg, 330, "f32", chunk=chunk, cuts=[20, 99, 101, 170] + list(range(250, 270)))
    check(ctx, cfg, 330, "bf16", chunk=chunk, cuts=[20, 99, 101, 170])


@pytest.mark.parametrize("window,keep", [(33, 7), (511, 0), (512, 130), (700, 1)])
def test_prompts_beyond_a_chunk(ctx, window, keep):
    """Several chunks of 512 around the window's size, kept rows that fill several tiles, then decoding."""
    cfg = lf.config([lf.attn(window=window, keep=keep, scale=0.6), lf.memory()])
    n = window + keep + 512 + 300
    check(ctx, cfg, n, "f32", cuts=[600, 602, 605, 800, 805] + list(range(n - 40, n)), chunk=512)


def test_largest_chunk_and_one_row_more(ctx):
    cfg = lf.config([lf.attn(window=70, scale=0.6), lf.memory(mlp=lf.moe(experts=9, top=2))], width=40)
    check(ctx, cfg, 2060, "f32", cuts=[2049, 2050])
    check(ctx, cfg, 2300, "f32", cuts=[100, 2270] + list(range(2280, 2300)))


def test_long_decoding(ctx):
    cfg = lf.config([lf.attn(window=20, keep=4, scale=0.6), lf.memory(mlp=lf.moe()), lf.attn(kv_from=0, window=31, keep=2)])
    check(ctx, cfg, 700, "f32", cuts=range(100, 700), chunk=64)   # the ring goes round many times


def test_long_decoding_with_a_graph_and_other_work_between(ctx):
    cfg = lf.config(MIXED)
    _, w, toks, want, _ = lf.clearest(cfg, 90, [0])
    m = lf.build(ctx, cfg, w, 128, DTYPE_F32)
    m.set_graph(True)
    got = [m.run_kv(toks[:30])]
    for i in range(30, 90):
        got.append(m.run_kv(toks[i:i + 1]))
        if i % 7 == 0:
            ctx.fill_lds()
            ctx.sync()
        if i == 60:
            m.set_graph(False)
        if i == 70:
            m.set_graph(True)
    m.close()
    verdict(np.concatenate(got), want, "f32")


def test_many_splits_without_a_window(ctx):
    cfg = lf.config([lf.attn(heads=2, kv_heads=1, dim=8, vdim=6, window=None, scale=0.7)], width=40)
    check(ctx, cfg, 2450, "f32", cuts=[2400] + list(range(2420, 2450)))


# ── keys that stand out ──

def spiked(cfg, w, query, key, gain=5.0):
    """Weights with which every head of layer 0 scores token `key` far above the rest when asked by token `query` (their
    rows of the embedding are large next to the position waves)."""
    m = cfg["layers"][0]["mixer"]
    rng = np.random.default_rng(99)
    u = rng.choice([-1.0, 1.0], m["dim"])
    x = w["embed"].astype(np.float64) * cfg["embedding"]["scale"]
    out = dict(w, **{"l0.mix.q.norm": np.ones(m["dim"], np.float32), "l0.mix.k.norm": np.ones(m["dim"], np.float32)})
    for name, heads, token in (("l0.mix.q", m["heads"], query), ("l0.mix.k", m["kv_heads"], key)):
        push = np.outer(np.tile(u, heads), x[token] / (x[token] @ x[token]))
        out[name] = lf.bf16(w[name] + gain * push)
    return out


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("window,keep", [(5, 3), (32, 31), (33, 64), (64, 65), (150, 1), (600, 40)])
def test_window_and_kept_edges(ctx, window, keep, dtype):
    """Token K stands out for token Q. K is planted at the last distance the window reaches, one further, as the last
    kept token and the first that is not, next to tile, split and chunk borders; the oracle's output differs clearly
    between seen and unseen."""
    cfg = lf.config([lf.attn(window=window, keep=keep, scale=0.9)], scale=25.0, mult=15.0)
    Q, K = 3, 4
    w = spiked(cfg, lf.weights(cfg, 5), Q, K)
    n = window + keep + 560
    base = tokens(cfg, n, 9)
    base[np.isin(base, (Q, K))] = 5
    cases = []
    for at in (keep + window - 1, keep + window, keep + window + 31, 511, 512, 513, n - 1):
        cases += [(at, at - window + 1), (at, at - window)]
    cases += [(n - 1, keep - 1), (n - 1, keep), (n - 1, 0), (keep + window + 40, keep - 1), (keep + window + 40, keep)]
    m = lf.build(ctx, cfg, w, n, DTYPES[dtype], 512 if window % 2 else 64)
    for at, key in cases:
        if not 0 <= key < at < n:
            continue
        toks = base[:at + 1].copy()
        toks[at], toks[key] = Q, K
        want, _ = lo.forward(cfg, w, toks)
        for how in ("prompt", "decoded"):
            m.reset_kv_cache()
            got = m.run_kv(toks) if how == "prompt" else feed(m, toks, [at])
            e_last, e_all = lf.error(got[-1:], want[-1:]), lf.error(got, want)
            assert e_last < MOST[dtype] and e_all < 2 * MOST[dtype], (window, keep, at, key, how, e_last, e_all)
        other = toks.copy()
        other[key] = 5
        gap = lf.error(lo.forward(cfg, w, other)[0][-1:], want[-1:])
        seen = at - key < window or key < keep
        assert gap > 0.2 if seen else gap < 1e-9, (window, keep, at, key, gap)
    m.close()


def test_a_far_token_in_the_memory(ctx):
    """One token's input gate opens wide, all others are nearly shut: hundreds of tokens later its value still decides,
    through chunk borders, portions and decoding."""
    cfg = lf.config([lf.memory(heads=2, dim=40, vdim=24, cap=10.0)], scale=25.0, mult=15.0)
    w = lf.weights(cfg, 8, gates=(-6.0, 8.0))
    x = w["embed"].astype(np.float64) * 25.0
    w["l0.mix.i"] = lf.bf16(w["l0.mix.i"] * 0.01 + np.outer(np.ones(2), x[7] / (x[7] @ x[7]) * 20.0))
    w["l0.mix.f"] = lf.bf16(w["l0.mix.f"] * 0.01)
    for at in (0, 1, 62, 63, 64, 65, 127, 200):
        toks = tokens(cfg, 420, 5)
        toks[toks == 7] = 8
        toks[at] = 7
        want, _ = lo.forward(cfg, w, toks)
        other = toks.copy()
        other[at] = 9
        assert lf.error(lo.forward(cfg, w, other)[0][-1:], want[-1:]) > 0.05
        run(ctx, cfg, w, toks, want, "f32", cuts=[at + 1, at + 2, 300, 301, 302] + list(range(400, 420)))
        run(ctx, cfg, w, toks, want, "bf16", cuts=[400])


def test_first_tokens(ctx):
    cfg = lf.config(MIXED)
    w = lf.weights(cfg)
    m = lf.build(ctx, cfg, w, 64, DTYPE_F32)
    for n in (1, 2, 3, 4, 8, 9):
        toks = tokens(cfg, n, 20 + n)
        want, _ = lo.forward(cfg, w, toks)
        for cuts in ((), (1,), range(1, n)):
            m.reset_kv_cache()
            verdict(feed(m, toks, cuts), want, "f32", f"{n} {list(cuts)}")
    m.close()


# ── what an earlier request leaves behind ──

def test_a_new_request_does_not_see_the_last_one(ctx):
    cfg = lf.config(MIXED)
    w = lf.weights(cfg)
    m = lf.build(ctx, cfg, w, 700, DTYPE_BF16, 64)
    a, b = tokens(cfg, 620, 1), tokens(cfg, 90, 2)
    alone = feed(m, b, [50, 52, 60, 61, 62])
    for _ in range(2):
        m.reset_kv_cache()
        feed(m, a, [600, 601], want=False)
        m.reset_kv_cache()
        assert m.kv_cache_len() == 0
        assert np.array_equal(feed(m, b, [50, 52, 60, 61, 62]), alone)
    m.reset_kv_cache()
    m.run_kv(a[:3], want_logits=False)
    m.reset_kv_cache()
    assert np.array_equal(feed(m, b, [50, 52, 60, 61, 62]), alone)
    m.close()


def test_cache_is_full_when_it_is(ctx):
    cfg = lf.config([lf.memory(), lf.attn()])
    m = lf.build(ctx, cfg, lf.weights(cfg), 20, DTYPE_F32)
    m.run_kv(tokens(cfg, 18), want_logits=False)
    with pytest.raises(HomuraError, match="full"):
        m.run_kv(tokens(cfg, 3))
    m.run_kv(tokens(cfg, 2), want_logits=False)
    with pytest.raises(HomuraError, match="full"):
        m.run_kv([1])
    m.close()


def test_prefill_pieces(ctx):
    cfg = lf.config([l for l in MIXED if not l["mlp"] or l["mlp"]["kind"] == "dense"][:1] + [lf.attn()])
    _, w, toks, want, _ = lf.clearest(cfg, 60, [2])
    m = lf.build(ctx, cfg, w, 64, DTYPE_BF16)
    errs = []
    for pieces in (1, 2, 3):
        m.set_prefill_pieces(pieces)
        m.reset_kv_cache()
        errs.append(lf.error(m.run_kv(toks), want))
    say(f"errors with 1, 2, 3 pieces: {errs}")
    assert errs[0] < LIMIT["bf16"] and max(errs[1:]) < errs[0]
    m.close()
    m = lf.build(ctx, lf.config(MIXED), lf.weights(lf.config(MIXED)), 64, DTYPE_BF16)
    with pytest.raises(HomuraError, match="pieces"):
        m.set_prefill_pieces(2)
    m.close()


# ── generation ──

def greedy_oracle(cfg, w, prompt, n):
    toks, margins = list(prompt), []
    for _ in range(n):
        row = lo.forward(cfg, w, toks)[0][-1]
        best = np.sort(row)
        margins.append(best[-1] - best[-2])
        toks.append(int(row.argmax()))
    return np.array(toks[len(prompt):]), min(margins)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("n_prompt", [1, 5, 40])
def test_greedy_generation(ctx, n_prompt, dtype):
    cfg = lf.config(MIXED)
    for seed in range(60, 90):     # a prompt whose picks are clear enough for the precision
        w = lf.weights(cfg, seed)
        prompt = tokens(cfg, n_prompt, seed)
        want, margin = greedy_oracle(cfg, w, prompt, 16)
        if margin > (1e-3 if dtype == "f32" else 0.04):
            break
    m = lf.build(ctx, cfg, w, 80, DTYPES[dtype])
    m.set_graph(True)
    if dtype == "bf16":
        m.set_prefill_pieces(3)
    assert np.array_equal(m.generate_greedy(prompt, 16), want)
    m.reset_kv_cache()
    assert np.array_equal(m.generate(prompt, 16, SamplingConfig(temperature=0.0, repetition_penalty=1.0)), want)
    m.close()


def test_an_end_token_takes_the_memories_back_to_where_generation_stopped(ctx):
    cfg = lf.config(MIXED)
    w, prompt = lf.weights(cfg, 3), tokens(cfg, 21, 3)
    m = lf.build(ctx, cfg, w, 120, DTYPE_F32)
    free = m.generate(prompt, 40, SamplingConfig(temperature=0.0, repetition_penalty=1.0))
    fresh = [i for i in range(40) if free[i] not in free[:i]]
    at = next((i for i in fresh if i >= 18), fresh[-1])
    m.reset_kv_cache()
    got = m.generate(prompt, 40, SamplingConfig(temperature=0.0, repetition_penalty=1.0), eos_token_id=int(free[at]))
    assert np.array_equal(got, free[:at])
    assert m.kv_cache_len() == len(prompt) + at
    more = tokens(cfg, 12, 8)
    cont = feed(m, more, [3, 4])
    want, _ = lo.forward(cfg, w, np.concatenate([prompt, free[:at], more]))
    m.close()
    verdict(cont, want[-12:], "f32")


def test_sampled_generation_follows_the_logits(ctx):
    cfg = lf.config(MIXED)
    w, prompt = lf.weights(cfg, 4), tokens(cfg, 12, 4)
    m = lf.build(ctx, cfg, w, 64, DTYPE_F32)
    sc = SamplingConfig(temperature=0.9, top_k=20, top_p=0.9, repetition_penalty=1.2)
    got = m.generate(prompt, 20, sc, seed=11)
    m.reset_kv_cache()
    rng, seen, row = Rng(11), [], m.run_kv(prompt)[-1]
    for t in got:
        assert sample_token_host(row, sc, seen, rng) == t
        seen.append(int(t))
        row = m.run_kv([t])[-1]
    m.close()


# ── from files ──

@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_model_directory_and_trace(ctx, tmp_path, dtype):
    cfg = lf.config(MIXED)
    short = "f32" if dtype == "float32" else "bf16"
    _, w, a, wa, _ = lf.clearest(cfg, 60, [6] if short == "f32" else range(6, 18))
    write_model(tmp_path / "m", cfg, w)
    m = homura_amd.load_model(ctx, tmp_path / "m", 100, dtype)
    assert isinstance(m, homura_amd.BlockModel) and (m.vocab_size, m.hidden_size, m.num_layers) == (101, 72, 6)
    b = a[:30]
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": a[:40].tolist(), "want": [39, 0]}], "end": []},
             {"step": 1, "entries": [{"id": "a", "tokens": a[40:43].tolist(), "want": []}], "end": []},
             {"step": 2, "entries": [{"id": "a", "tokens": a[43:].tolist(), "want": [16]}], "end": ["a"]},
             {"step": 3, "entries": [{"id": "b", "tokens": b.tolist(), "want": list(range(30))}], "end": ["b"]}]
    trace.replay(m, [json.dumps(s) for s in steps], tmp_path, lambda s: say(s))
    m.close()
    row = lambda n: np.fromfile(tmp_path / f"{n}.f32", "<f4").reshape(-1, 101)
    for got, want in ((row(0), wa[[39, 0]]), (row(2), wa[[59]]), (row(3), wa[:30])):
        assert lf.error(got, want) < LIMIT[short]


def test_files_and_sizes_that_do_not_fit_are_named(ctx, tmp_path):
    cfg = lf.config([lf.memory(), lf.attn(mlp=lf.moe())])
    w = lf.weights(cfg)
    write_model(tmp_path / "a", cfg, w, drop=("l1.mlp.e3.up",))
    with pytest.raises(HomuraError, match="l1.mlp.e3.up"):
        homura_amd.load_model(ctx, tmp_path / "a", 32)
    write_model(tmp_path / "b", cfg, w, reshape={"l0.mix.i": (72, 3)})
    with pytest.raises(HomuraError, match="l0.mix.i"):
        homura_amd.load_model(ctx, tmp_path / "b", 32)
    for layer, message in ((lf.attn(dim=257), "256"), (lf.memory(dim=1025), "1024"), (lf.attn(mlp=lf.moe(experts=1025, top=1)), "experts")):
        with pytest.raises(HomuraError, match=message):
            homura_amd.BlockModel(ctx, lf.config([layer]))
