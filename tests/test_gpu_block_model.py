"""List-of-layers (Nokuvik) models on the GPU against the numpy oracle: every mechanism alone, prompts in one piece
and in portions, decoding, windows and their edges, reuse of the cache, generation. `f32` runs everything in 32 bits
and is held to 2e-5 of the logits' spread; `bf16` is the serving precision."""
from __future__ import annotations

import ctypes as C
import json

import numpy as np
import pytest

import block_fixture as bf
import ckpt_writers as cw
import homura_amd
import nokuvik_oracle as no
from homura_amd import synth, trace
from homura_amd.runtime import DTYPE_BF16, DTYPE_F32, HomuraError, Rng, SamplingConfig, sample_token_host

pytestmark = pytest.mark.gpu

DTYPES = {"f32": DTYPE_F32, "bf16": DTYPE_BF16}
LIMIT = {"f32": 2e-5, "bf16": 0.06}


def say(msg):
    print(f"[block model] {msg}", flush=True)


def tokens(cfg, n, seed=7):
    return np.random.default_rng(seed).integers(0, cfg["vocab"], n)


def feed(m, toks, cuts, want=True):
    """Runs toks in portions ending at `cuts` (and at the end); all logits."""
    out, at = [], 0
    for end in list(cuts) + [len(toks)]:
        if end > at:
            out.append(m.run_kv(toks[at:end], want_logits=want))
            at = end
    return np.concatenate(out) if want else None


def check(ctx, cfg, n, dtype, seed=0, max_len=None, cuts=(), prefill_min=8, w=None, chunk=None):
    say(f"{n} tokens, {dtype}, cuts {list(cuts)[:6]}, {json.dumps(cfg)[:160]}")
    w = bf.weights(cfg, seed) if w is None else w
    toks = tokens(cfg, n, seed + 1)
    want, _ = no.forward(cfg, w, toks)
    m = bf.build(ctx, cfg, w, max_len or n, DTYPES[dtype], chunk)
    m.set_prefill_min(prefill_min)
    got = feed(m, toks, cuts)
    m.close()
    err = bf.error(got, want)
    say(f"error {err:.2e}")
    assert err < LIMIT[dtype]
    return got, want


# ── each mechanism alone, in a prompt and token by token ──

ONE_LAYER = {
    "latent": bf.attn(),
    "latent_ff": bf.attn(ff=37),
    "latent_part_rotated": bf.attn(rot_dim=14, rot_dims=6),
    "latent_one_head": bf.attn(heads=1, dim=1, rot_dim=2, vdim=1, q_rank=3, kv_rank=2, window=2),
    "latent_many_heads": bf.attn(heads=21, dim=9, rot_dim=4, vdim=5, q_rank=31, kv_rank=33),
    "latent_wide_rank": bf.attn(heads=2, kv_rank=530, q_rank=70),
    "latent_widest_rank": bf.attn(heads=2, kv_rank=1010),
    "latent_window_1": bf.attn(window=1),
    "latent_128": bf.attn(heads=2, dim=70, rot_dim=30, vdim=90),
    "latent_192": bf.attn(heads=2, dim=128, rot_dim=64, vdim=128),
    "latent_256": bf.attn(heads=2, dim=150, rot_dim=60, vdim=140),
    "latent_vdim_64": bf.attn(heads=2, dim=40, rot_dim=24, vdim=64),
    "scan": bf.scan(),
    "scan_ff": bf.scan(ff=50),
    "scan_one_tap": bf.scan(conv=1, state=1, dt_rank=1),
    "scan_16_states": bf.scan(state=16, inner=64),
    "scan_wide": bf.scan(inner=130, conv=6, dt_rank=40, state=33),
    "scan_100_states": bf.scan(state=100, dt_rank=33),
    "recurrence": bf.recurrence(),
    "recurrence_ff": bf.recurrence(ff=96),
    "recurrence_one_block": bf.recurrence(width=50, conv=1, blocks=1),
    "recurrence_small_blocks": bf.recurrence(width=66, conv=5, blocks=22),
    "recurrence_wide_blocks": bf.recurrence(width=600, conv=2, blocks=2),
}


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("name", list(ONE_LAYER))
def test_one_mechanism(ctx, name, dtype):
    if name == "latent_one_head" and dtype == "bf16":
        pytest.skip("a norm over two values takes their bf16 rounding to any size")
    cfg = bf.config([ONE_LAYER[name]])
    check(ctx, cfg, 70, dtype)
    check(ctx, cfg, 45, dtype, prefill_min=0)


@pytest.mark.parametrize("width", [40, 96, 260, 1100])
def test_other_widths(ctx, width):
    cfg = bf.config([bf.scan(ff=33), bf.attn(ff=70), bf.recurrence()], width=width, vocab=517, eps=1e-6,
                    loop={"start": 1, "stop": 2, "times": 2})
    check(ctx, cfg, 40, "f32")
    check(ctx, cfg, 20, "f32", prefill_min=0)


def test_heads_too_wide_for_the_prompt_pass_take_decode_steps(ctx):
    cfg = bf.config([bf.attn(heads=2, dim=250, rot_dim=20, vdim=30)])
    w = bf.weights(cfg)
    m = bf.build(ctx, cfg, w, 30, DTYPE_F32)
    toks = tokens(cfg, 30)
    assert bf.error(m.run_kv(toks), no.forward(cfg, w, toks)[0]) < LIMIT["f32"]
    with pytest.raises(HomuraError, match="256"):
        m.prefill(toks)
    m.close()


# ── order of layers, loops ──

MIXED = [bf.attn(ff=90), bf.scan(), bf.recurrence(), bf.scan(ff=41, state=17)]
LOOPS = {"none": None, "all": {"start": 0, "stop": 4, "times": 2}, "middle": {"start": 1, "stop": 3, "times": 3},
         "tail_once": {"start": 2, "stop": 4, "times": 1}, "first": {"start": 0, "stop": 1, "times": 4}}


@pytest.mark.parametrize("loop", list(LOOPS))
def test_loops(ctx, loop):
    cfg = bf.config(MIXED, loop=LOOPS[loop])
    check(ctx, cfg, 60, "f32", cuts=(33, 34, 35, 36, 50))
    check(ctx, cfg, 60, "bf16", cuts=(33, 34, 35, 36, 50))


def test_residual_behind_every_layer_run(ctx):
    cfg = bf.config(MIXED, loop=LOOPS["middle"])
    w, toks = bf.weights(cfg), tokens(cfg, 50)
    _, trail = no.forward(cfg, w, toks)
    m = bf.build(ctx, cfg, w, 64, DTYPE_F32)
    m.capture_residuals()
    m.prefill(toks)
    got = m.captured_residuals(len(trail), len(toks))
    m.close()
    for i, (g, t) in enumerate(zip(got, trail)):
        assert bf.error(g, t) < 1e-5, f"layer run {i}"


# ── portions ──

@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("size", [2, 3, 7, 8, 9, 31, 64])
def test_portions(ctx, size, dtype):
    cfg = bf.config(MIXED, loop=LOOPS["all"])
    check(ctx, cfg, 130, dtype, cuts=range(size, 130, size))


def test_portions_of_changing_size_then_single_tokens(ctx):
    cfg = bf.config(MIXED, loop=LOOPS["middle"])
    cuts = list(np.cumsum([1, 40, 2, 8, 3, 17, 5, 9, 2, 2, 30])) + list(range(120, 150))
    check(ctx, cfg, 150, "f32", cuts=cuts)


@pytest.mark.parametrize("window", [33, 511, 512, 513, 700])
def test_prompts_beyond_a_chunk_and_around_the_ring(ctx, window):
    """A prompt of several chunks of 512, the window below, at and above the chunk's size, then decoding: the ring of
    cache rows (window - 1 + 512) goes round, and keys come from earlier chunks, portions and steps."""
    cfg = bf.config([bf.attn(window=window, scale=0.6), bf.recurrence(), bf.scan()])
    n = window - 1 + 512 + 300
    check(ctx, cfg, n, "f32", cuts=[600, 602, 605, 800, 805] + list(range(n - 40, n)), chunk=512)


@pytest.mark.parametrize("chunk", [16, 33, 100])
def test_small_chunks(ctx, chunk):
    cfg = bf.config(MIXED, loop=LOOPS["all"])
    check(ctx, cfg, 210, "f32", chunk=chunk)
    check(ctx, cfg, 210, "bf16", cuts=(20, 99, 101, 170), chunk=chunk)


def test_largest_chunk_and_one_row_more(ctx):
    cfg = bf.config([bf.attn(window=70, scale=0.6), bf.recurrence(), bf.scan()], width=40)
    check(ctx, cfg, 2060, "f32", cuts=[2049, 2050])
    check(ctx, cfg, 2300, "f32", cuts=[100, 2270] + list(range(2280, 2300)))


def test_chunk_size_limits(ctx):
    m = homura_amd.BlockModel(ctx, bf.config(MIXED))
    for rows in (15, 2049):
        with pytest.raises(HomuraError, match="chunk"):
            m.set_prefill_chunk(rows)
    m.close()


def test_long_decoding(ctx):
    cfg = bf.config([bf.attn(window=20, scale=0.6), bf.scan(), bf.recurrence()])
    check(ctx, cfg, 700, "f32", cuts=range(100, 700), chunk=64)   # the ring goes round many times


def test_long_decoding_with_a_graph_and_other_work_between(ctx):
    cfg = bf.config(MIXED, loop=LOOPS["all"])
    w, toks = bf.weights(cfg), tokens(cfg, 90)
    want, _ = no.forward(cfg, w, toks)
    m = bf.build(ctx, cfg, w, 128, DTYPE_F32)
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
    assert bf.error(np.concatenate(got), want) < LIMIT["f32"]


def test_many_splits_of_a_wide_window(ctx):
    """A window of more rows than 64 splits of one tile: tiles follow one another inside a split."""
    cfg = bf.config([bf.attn(heads=2, dim=8, rot_dim=4, vdim=6, q_rank=20, kv_rank=16, window=2300, scale=1.0)], width=40)
    check(ctx, cfg, 2450, "f32", cuts=[2400] + list(range(2420, 2450)))


# ── keys that stand out ──

def spiked(cfg, w, query, key, layer=0, gain=18.0):
    """Weights in which every head of `layer` scores token `key` far above the rest when asked by token `query`
    (ahead of any other layer: the residual is the embedding)."""
    m, p = cfg["layers"][layer]["mixer"], f"l{layer}."
    eps = cfg["norm"]["eps"]
    x = w["embed"].astype(np.float64) * cfg["embedding"]["scale"]
    h = no.rms_norm(x, w[p + "norm1"].astype(np.float64), eps)
    q = no.rms_norm(h[query] @ w[p + "mix.dq"].T, w[p + "mix.dq.norm"], eps) @ w[p + "mix.uq"].T
    q = q.reshape(m["heads"], -1)[:, :m["dim"]]
    c = no.rms_norm((h[key] @ w[p + "mix.dkv"].T)[:m["kv_rank"]], w[p + "mix.dkv.norm"], eps)
    uk = w[p + "mix.uk"].astype(np.float64).reshape(m["heads"], m["dim"], -1)
    for a in range(m["heads"]):
        uk[a] += gain / m["scale"] * np.outer(q[a] / (q[a] @ q[a]), c / (c @ c))
    return dict(w, **{p + "mix.uk": bf.bf16(uk.reshape(w[p + "mix.uk"].shape))})


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("window", [5, 32, 33, 64, 150, 600])
def test_window_edges(ctx, window, dtype):
    """Token K stands out for token Q. K is planted at the last distance the window reaches, one further, and next
    to tile, split and chunk borders; the oracle's output differs clearly between seen and unseen."""
    cfg = bf.config([bf.attn(window=window)])
    Q, K = 3, 4
    w = spiked(cfg, bf.weights(cfg, 5), Q, K)
    n = window + 560
    base = tokens(cfg, n, 9)
    base[np.isin(base, (Q, K))] = 5
    ends = [window - 1, window, window + 31, 511, 512, 513, n - 1]
    for far in (window - 1, window):          # just seen, just not
        for at in ends:
            if at - far < 0:
                continue
            toks = base[:at + 1].copy()
            toks[at], toks[at - far] = Q, K
            want, _ = no.forward(cfg, w, toks)
            m = bf.build(ctx, cfg, w, n, DTYPES[dtype], 512 if window % 2 else None)
            for how in ("prompt", "decoded"):
                m.reset_kv_cache()
                got = m.run_kv(toks) if how == "prompt" else feed(m, toks, [at])
                e_last, e_all = bf.error(got[-1:], want[-1:]), bf.error(got, want)
                assert e_last < LIMIT[dtype] and e_all < 2 * LIMIT[dtype], (window, far, at, how, e_last, e_all)
            m.close()
            other = toks.copy()
            other[at - far] = 5
            gap = bf.error(no.forward(cfg, w, other)[0][-1:], want[-1:])
            assert gap > 0.3 if far == window - 1 else gap < 1e-9, (window, far, at, gap)


def test_first_tokens(ctx):
    cfg = bf.config(MIXED, loop=LOOPS["all"])
    w = bf.weights(cfg)
    m = bf.build(ctx, cfg, w, 64, DTYPE_F32)
    for n in (1, 2, 3, 4, 8, 9):
        toks = tokens(cfg, n, 20 + n)
        want, _ = no.forward(cfg, w, toks)
        for cuts in ((), (1,), range(1, n)):
            m.reset_kv_cache()
            assert bf.error(feed(m, toks, cuts), want) < LIMIT["f32"], (n, list(cuts))
    m.close()


# ── what an earlier request leaves behind ──

def test_a_new_request_does_not_see_the_last_one(ctx):
    cfg = bf.config(MIXED, loop=LOOPS["middle"])
    w = bf.weights(cfg)
    m = bf.build(ctx, cfg, w, 700, DTYPE_BF16)
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


def test_a_prompt_without_logits_leaves_the_same_state(ctx):
    """The feed-forward behind the last mixer has no reader then."""
    cfg = bf.config([bf.attn(), bf.recurrence(), bf.scan(ff=50)])
    m = bf.build(ctx, cfg, bf.weights(cfg), 128, DTYPE_BF16)
    a, rows = tokens(cfg, 60), []
    for want in (True, False):
        m.reset_kv_cache()
        m.prefill(a[:40], want_logits=want)
        m.prefill(a[40:57], want_logits=want)
        rows.append(np.concatenate([m.run_kv(a[i:i + 1]) for i in range(57, 60)]))
    assert np.array_equal(rows[0], rows[1])
    m.close()


def test_cache_is_full_when_it_is(ctx):
    cfg = bf.config([bf.scan(), bf.attn()])
    m = bf.build(ctx, cfg, bf.weights(cfg), 20, DTYPE_F32)
    m.run_kv(tokens(cfg, 18), want_logits=False)
    with pytest.raises(HomuraError, match="full"):
        m.run_kv(tokens(cfg, 3))
    m.run_kv(tokens(cfg, 2), want_logits=False)
    with pytest.raises(HomuraError, match="full"):
        m.run_kv([1])
    m.close()


def test_prefill_pieces(ctx):
    cfg = bf.config(MIXED)
    w, toks = bf.weights(cfg), tokens(cfg, 60)
    want, _ = no.forward(cfg, w, toks)
    m = bf.build(ctx, cfg, w, 64, DTYPE_BF16)
    errs = []
    for pieces in (1, 2, 3):
        m.set_prefill_pieces(pieces)
        m.reset_kv_cache()
        errs.append(bf.error(m.run_kv(toks), want))
    say(f"errors with 1, 2, 3 pieces: {errs}")
    assert errs[0] < LIMIT["bf16"] and max(errs[1:]) < errs[0]
    m.close()
    m = bf.build(ctx, cfg, w, 64, DTYPE_F32)
    with pytest.raises(HomuraError, match="pieces"):
        m.set_prefill_pieces(2)
    with pytest.raises(HomuraError, match="not available"):
        m._check(m.lib.hm_model_set_whole_step(m.h, 1))
    m.close()


# ── generation ──

def greedy_oracle(cfg, w, prompt, n):
    toks, margins = list(prompt), []
    for _ in range(n):
        row = no.forward(cfg, w, toks)[0][-1]
        best = np.sort(row)
        margins.append(best[-1] - best[-2])
        toks.append(int(row.argmax()))
    return np.array(toks[len(prompt):]), min(margins)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("n_prompt", [1, 5, 40])
def test_greedy_generation(ctx, n_prompt, dtype):
    cfg = bf.config(MIXED, loop=LOOPS["all"])
    for seed in range(60, 80):     # a prompt whose picks are clear enough for the precision
        w = bf.weights(cfg, seed)
        prompt = tokens(cfg, n_prompt, seed)
        want, margin = greedy_oracle(cfg, w, prompt, 16)
        if margin > (1e-3 if dtype == "f32" else 0.04):
            break
    m = bf.build(ctx, cfg, w, 80, DTYPES[dtype])
    m.set_graph(True)
    if dtype == "bf16":
        m.set_prefill_pieces(3)
    assert np.array_equal(m.generate_greedy(prompt, 16), want)
    m.reset_kv_cache()
    assert np.array_equal(m.generate(prompt, 16, SamplingConfig(temperature=0.0, repetition_penalty=1.0)), want)
    m.close()


def test_an_end_token_takes_recurrent_state_back_to_where_generation_stopped(ctx):
    """Steps run ahead of the host in chunks; those behind an end-of-sequence token must leave nothing in the states,
    the convolutions and the window."""
    cfg = bf.config(MIXED, loop=LOOPS["middle"])
    w, prompt = bf.weights(cfg, 3), tokens(cfg, 21, 3)
    m = bf.build(ctx, cfg, w, 120, DTYPE_F32)
    free = m.generate(prompt, 40, SamplingConfig(temperature=0.0, repetition_penalty=1.0))
    at = next(i for i in range(18, 40) if free[i] not in free[:i]) if any(free[i] not in free[:i] for i in range(18, 40)) else \
        max(i for i in range(40) if free[i] not in free[:i])
    m.reset_kv_cache()
    got = m.generate(prompt, 40, SamplingConfig(temperature=0.0, repetition_penalty=1.0), eos_token_id=int(free[at]))
    assert np.array_equal(got, free[:at])
    assert m.kv_cache_len() == len(prompt) + at
    more = tokens(cfg, 12, 8)
    cont = feed(m, more, [3, 4])
    whole = np.concatenate([prompt, free[:at], more])
    want, _ = no.forward(cfg, w, whole)
    m.close()
    assert bf.error(cont, want[-12:]) < LIMIT["f32"]


def test_sampled_generation_follows_the_logits(ctx):
    cfg = bf.config(MIXED)
    w, prompt = bf.weights(cfg, 4), tokens(cfg, 12, 4)
    m = bf.build(ctx, cfg, w, 64, DTYPE_F32)
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

def write_model(path, cfg, w, drop=(), reshape=None):
    path.mkdir(exist_ok=True)
    tensors = {k: ("BF16", (reshape or {}).get(k, v.shape), synth.f32_to_bf16_rne(v).tobytes()) for k, v in w.items() if k not in drop}
    (path / "config.json").write_text(json.dumps(cfg))
    (path / "model.safetensors").write_bytes(cw.safetensors_bytes(tensors))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_model_directory_and_trace(ctx, tmp_path, dtype):
    cfg = bf.config(MIXED, loop=LOOPS["all"])
    w = bf.weights(cfg, 6)
    write_model(tmp_path / "m", cfg, w)
    m = homura_amd.load_model(ctx, tmp_path / "m", 100, dtype)
    assert isinstance(m, homura_amd.BlockModel) and (m.vocab_size, m.hidden_size, m.num_layers) == (101, 72, 4)
    a, b = tokens(cfg, 60, 1), tokens(cfg, 30, 2)
    wa, wb = no.forward(cfg, w, a)[0], no.forward(cfg, w, b)[0]
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": a[:40].tolist(), "want": [39, 0]}], "end": []},
             {"step": 1, "entries": [{"id": "a", "tokens": a[40:43].tolist(), "want": []}], "end": []},
             {"step": 2, "entries": [{"id": "a", "tokens": a[43:].tolist(), "want": [16]}], "end": ["a"]},
             {"step": 3, "entries": [{"id": "b", "tokens": b.tolist(), "want": list(range(30))}], "end": ["b"]}]
    trace.replay(m, [json.dumps(s) for s in steps], tmp_path, lambda s: say(s))
    m.close()
    row = lambda n: np.fromfile(tmp_path / f"{n}.f32", "<f4").reshape(-1, 101)
    limit = LIMIT["f32" if dtype == "float32" else "bf16"]
    assert bf.error(row(0), wa[[39, 0]]) < limit and bf.error(row(2), wa[[59]]) < limit and bf.error(row(3), wb) < limit


def test_files_that_do_not_fit_are_named(ctx, tmp_path):
    cfg = bf.config([bf.recurrence(), bf.scan()])
    w = bf.weights(cfg)
    write_model(tmp_path / "a", cfg, w, drop=("l0.mix.ra",))
    with pytest.raises(HomuraError, match="l0.mix.ra"):
        homura_amd.load_model(ctx, tmp_path / "a", 32)
    write_model(tmp_path / "b", cfg, w, reshape={"l1.mix.o": (48, 72)})
    with pytest.raises(HomuraError, match="l1.mix.o"):
        homura_amd.load_model(ctx, tmp_path / "b", 32)
    write_model(tmp_path / "c", dict(cfg, architecture="Unheard"), w)
    with pytest.raises(HomuraError, match="Unheard"):
        homura_amd.load_model(ctx, tmp_path / "c", 32)
    m = homura_amd.BlockModel(ctx, cfg)
    with pytest.raises(HomuraError, match="missing weight"):
        m.finalize(32)
    m.close()


# q latents of two, four and eight vectors a lane, cache rows of both, parts of rows that are no whole vectors (the workgroup a row);
# queries that turn where they lie (192 = 128 + 64 wide), with a part that does not turn, and wider rows than the projection's;
# keys and values written by their product, with columns behind them (head rows of 64 / 128), a head's end inside a tile, and 24 rows of few
LATENTS = {
    "turned_in_place": dict(heads=5, dim=128, rot_dim=64, rot_dims=64, vdim=128, q_rank=96, kv_rank=64),
    "half_turned": dict(heads=3, dim=128, rot_dim=64, rot_dims=24, vdim=120, q_rank=1000, kv_rank=192),
    "wider_rows": dict(heads=7, dim=24, rot_dim=8, rot_dims=8, vdim=40, q_rank=260, kv_rank=600),
    "wide_latents": dict(heads=2, dim=64, rot_dim=64, rot_dims=48, vdim=64, q_rank=1030, kv_rank=1024),
    "widest_latents": dict(heads=2, dim=64, rot_dim=64, rot_dims=64, vdim=64, q_rank=1540, kv_rank=128),
    "odd_parts": dict(heads=3, dim=26, rot_dim=6, rot_dims=6, vdim=30, q_rank=70, kv_rank=64),
}


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("name", list(LATENTS))
def test_latent_rows_of_a_prompt(ctx, name, dtype):
    cfg = bf.config([bf.attn(window=150, **LATENTS[name])])
    check(ctx, cfg, 333, dtype, cuts=(24, 190))


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("n", [70, 300])
def test_gate_rows_from_slices_and_whole(ctx, n, dtype):
    """The gates of the scan and the recurrence straight from their projection, and from the convolution where it came in K slices (1100 wide)."""
    routes = (C.c_longlong * 3)()
    for width in (1100, 96):
        ctx._check(ctx.lib.hm_test_routes(ctx.h, routes))
        whole, sliced = routes[1:]
        cfg = bf.config([bf.scan(inner=64, state=16), bf.scan(inner=130, state=33), bf.recurrence(), bf.recurrence(width=66, blocks=2)], width=width)
        check(ctx, cfg, n, dtype, cuts=(n // 3,))
        ctx._check(ctx.lib.hm_test_routes(ctx.h, routes))
        assert (routes[1] > whole, routes[2] > sliced) == (width == 96, width == 1100)


# one to four wavefronts a row, the last of them part of the way; one round of rows, several with a last one of few rows; the paired, the
# plain and the convolution epilogue behind one norm and two
@pytest.mark.parametrize("width,ff", [(72, 4107), (520, 33), (1000, 4200), (1024, 8300), (1100, 37), (1536, 4500), (1800, 8200), (2048, 37)])
def test_decode_products_behind_a_norm(ctx, width, ff):
    cfg = bf.config([bf.scan(inner=64, state=16, ff=ff), bf.recurrence(width=66, blocks=2, ff=ff), bf.attn(heads=3)], width=width)
    check(ctx, cfg, 9, "bf16", prefill_min=0)


# one to eight vectors a lane, in one slice and in several, ranks that fill no whole wavefront, one and three pieces
@pytest.mark.parametrize("q_rank,rank,rot,parts,pieces,n,past", [(768, 512, 64, 1, 1, 33, 0), (100, 36, 8, 1, 3, 5, 2), (512, 132, 128, 1, 1, 7, 0),
                                                                  (2048, 1024, 64, 1, 1, 9, 3), (1536, 512, 64, 1, 3, 2, 0), (4, 4, 0, 1, 1, 1, 0),
                                                                  (256, 512, 32, 3, 1, 6, 1), (1024, 260, 16, 8, 3, 4, 0)])
def test_latent_rows_have_the_same_bits_from_either_kernel(ctx, q_rank, rank, rot, parts, pieces, n, past):
    """A wavefront a row, and a workgroup a row (which a row stride of no whole vectors takes; the decode step writes its cache row with the same
    code): the same values in another place give the same bits."""
    rng = np.random.default_rng(q_rank + rank + parts)
    pad = lambda w: (w + 31) // 32 * 32
    q_pad, wide = pad(q_rank), pad(q_rank) + rank + rot
    values = rng.standard_normal((parts, n, wide)).astype(np.float32)
    q_norm, kv_norm = (1 + 0.1 * rng.standard_normal((2, max(q_pad, pad(rank))))).astype(np.float32)
    cos, sin = rng.standard_normal((2, past + n, max(rot, 4))).astype(np.float32)
    dev = [ctx.to_device(v) for v in (q_norm, kv_norm, cos.reshape(-1)[:(past + n) * max(rot, 4)], sin.reshape(-1)[:(past + n) * max(rot, 4)])]
    got = []
    for ld in (wide + 3 & ~3, (wide + 3 & ~3) + 1):
        down = np.full((parts, n, ld), np.nan, np.float32)
        down[:, :, :wide] = values
        d = ctx.to_device(down)
        q, ring = (ctx.to_device(np.full(size + 64, 0x7B7B, np.uint16)) for size in (n * pieces * q_pad, (past + n) * pieces * (pad(rank) + pad(rot))))
        ctx._check(ctx.lib.hm_test_latent_rows(ctx.h, d.ptr, ld, parts, *(b.ptr for b in dev), q_rank, rank, rot, pieces, n, past, 1e-6, q.ptr, ring.ptr))
        got.append((q.download(np.uint16), ring.download(np.uint16)))
        for b in (d, q, ring):
            b.free()
    for b in dev:
        b.free()
    for wave, group in zip(*got):
        assert np.all(wave[-64:] == 0x7B7B) and np.array_equal(wave, group)
