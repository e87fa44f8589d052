"""What this framework is measured on: whole requests to its decoders through DecoderModel.generate / prefill / run_kv,
and the kernel-level entry points that a C or Rust caller drives directly.

A model is loaded once and kept (weights of one fixed random draw per model, as a checkpoint would be), and requests with
prompts of their own are put to it; every request starts on an empty cache. The embedding row of token t points where the
output row of token t + 1 does, so that the next token has the clear lead it has in a trained model: picks do not hang on
the last bits of a logit, and the sampler meets a peaked distribution.
"""
import ctypes
import dataclasses
import math
import zlib

import numpy as np
import torch

from homura_amd import (DTYPE_BF16, DTYPE_Q4_0, DTYPE_Q4_K, DTYPE_Q6_K, DTYPE_Q8_0, BlockModel, Context, HfModel, synth_model)
from homura_amd.runtime import SamplingConfig

MAX_SEQ = 8192
BLOCK = {"q8_0": (32, 34), "q4_0": (32, 18), "q4_k": (256, 144), "q6_k": (256, 210)}  # weights and bytes of a block
CODE = {"bf16": DTYPE_BF16, "q8_0": DTYPE_Q8_0, "q4_0": DTYPE_Q4_0, "q4_k": DTYPE_Q4_K, "q6_k": DTYPE_Q6_K}
GREEDY = SamplingConfig(temperature=0.0, repetition_penalty=1.0)
DEFAULT = SamplingConfig()


# ── the cases ──

def listed():
    return [
        # One weight product of a caller that keeps raw GGUF blocks: TinyLlama's gate, one row (small: latency counts).
        {"name": "gemv-q8_0-2048x5632", "op": "gemv", "fmt": "q8_0", "k": 2048, "n": 5632},
        # A prompt chunk through one projection in the weight layout the reference hands its kernels.
        {"name": "gemm-512x2048x8192", "op": "gemm", "nk": False, "m": 512, "k": 2048, "n": 8192},
        # Attention of a batch of eight sequences over long caches.
        {"name": "attention-8x12q2kv-4096", "op": "attention", "b": 8, "h": 12, "kvh": 2, "hd": 128, "len": 4096},
        # The everyday chat answer: a short question, a sampled answer with the default settings.
        {"name": "0.6b-bf16-answer", "op": "reply", "model": "qwen3-0.6b", "fmt": "bf16", "prompt": 24, "new": 64, "sampled": True},
        # Time to the first token of an ordinary prompt.
        {"name": "0.6b-bf16-prompt-512", "op": "prompt", "model": "qwen3-0.6b", "fmt": "bf16", "prompt": 512},
        # A long document and a short answer about it.
        {"name": "0.6b-bf16-document", "op": "reply", "model": "qwen3-0.6b", "fmt": "bf16", "prompt": 6001, "new": 16, "sampled": False},
        # A Q4_K_M file, as most GGUF users load one.
        {"name": "0.6b-q4_k_m-answer", "op": "reply", "model": "qwen3-0.6b", "fmt": "q4_k_m", "prompt": 181, "new": 32, "sampled": True},
        # A Q8_0 file reading a page.
        {"name": "0.6b-q8_0-prompt-1000", "op": "prompt", "model": "qwen3-0.6b", "fmt": "q8_0", "prompt": 1000},
        # A short turn on the smallest listed model: launches and small row counts.
        {"name": "0.5b-bf16-turn", "op": "prompt", "model": "qwen2.5-0.5b", "fmt": "bf16", "prompt": 37},
        # A larger model without a whole-step launch.
        {"name": "1.5b-bf16-answer", "op": "reply", "model": "qwen2.5-1.5b", "fmt": "bf16", "prompt": 700, "new": 32, "sampled": False},
        # The list-of-layers families: a prompt through scans, recurrences and latent attention ...
        {"name": "nokuvik-prompt-2048", "op": "prompt", "model": "nokuvik-1024", "fmt": "bf16", "prompt": 2048},
        # ... and an answer through matrix memories and mixtures of experts.
        {"name": "ludalix-answer", "op": "reply", "model": "ludalix-1024", "fmt": "bf16", "prompt": 300, "new": 32, "sampled": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["gemv", "gemm", "attention", "reply", "reply", "reply", "prompt", "prompt", "prompt"])
    if op == "gemv":
        fmt = rng.choice(["bf16", "q8_0", "q4_0", "q4_k", "q6_k"])
        return {"op": op, "fmt": fmt, "k": 256 * _log(rng, 3, 16), "n": _log(rng, 896, 32000)}
    if op == "gemm":
        return {"op": op, "nk": rng.random() < 0.5, "m": _log(rng, 16, 2048), "k": 64 * _log(rng, 8, 96), "n": 8 * _log(rng, 64, 1024)}
    if op == "attention":
        h, kvh, hd = rng.choice([(16, 8, 128), (14, 2, 64), (32, 4, 64), (12, 2, 128), (32, 32, 64)])
        return {"op": op, "b": rng.randint(1, 8), "h": h, "kvh": kvh, "hd": hd, "len": _log(rng, 32, 8000)}
    model = rng.choice(["qwen3-0.6b"] * 4 + ["qwen2.5-0.5b", "tinyllama-1.1b", "qwen2.5-1.5b", "nokuvik-1024", "ludalix-1024"])
    fmts = {"qwen2.5-0.5b": ["bf16", "q8_0", "q4_0"], "nokuvik-1024": ["bf16"], "ludalix-1024": ["bf16"]}
    case = {"op": op, "model": model, "fmt": rng.choice(fmts.get(model, ["bf16", "q8_0", "q4_0", "q4_k_m"]))}
    case["prompt"] = _log(rng, 2, 6000 if model == "qwen3-0.6b" else 2000)
    if op == "reply":
        case.update(new=rng.randint(4, 32), sampled=rng.random() < 0.5)
    return case


# ── values ──

def _normal(name, shape, scale, mean=0.0):
    g = torch.Generator("cuda").manual_seed(zlib.crc32(name.encode()))
    return torch.randn(shape, generator=g, device="cuda") * scale + mean


def _blocks(name, fmt, rows, k, std):
    """Raw GGUF blocks [rows][k / block] of weights around zero with the standard deviation `std`."""
    g = torch.Generator("cuda").manual_seed(zlib.crc32(name.encode()))
    n, (_, size) = rows * k // BLOCK[fmt][0], BLOCK[fmt]
    b = torch.randint(0, 256, (n, size), generator=g, device="cuda", dtype=torch.uint8)
    spread = {"q8_0": 73.9, "q4_0": 4.61, "q4_k": 4.61 * 36.5, "q6_k": 18.5 * 73.9}[fmt]
    d = std / spread * (0.8 + 0.4 * torch.rand(n, generator=g, device="cuda"))

    def half(x):
        return x.to(torch.float16).view(torch.uint8).reshape(n, 2)
    if fmt == "q4_k":  # minima of seven and a half steps a sub-block
        b[:, 8:12] = b[:, 4:8]
        b[:, 12:16] = (b[:, 12:16] & 15) * 17
        b[:, 0:2], b[:, 2:4] = half(d), half(7.5 * d)
    elif fmt == "q6_k":
        b[:, 208:210] = half(d)
    else:
        if fmt == "q4_0":  # quants 1 to 15 around eight, as a quantiser of signed values leaves them
            b = torch.where((b & 15) == 0, b + 8, b)
            b = torch.where((b >> 4) == 0, b + 128, b)
        b[:, 0:2] = half(d)
    return b.reshape(rows, -1)


def _weights(raw, fmt, k):
    """The float64 matrix [rows, k] that raw blocks or bf16 values stand for."""
    if fmt == "bf16":
        return raw.double()
    rows, b = raw.shape[0], raw.reshape(-1, BLOCK[fmt][1])

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()
    if fmt == "q8_0":
        w = b[:, 2:].contiguous().view(torch.int8).double() * half(0)
    elif fmt == "q4_0":
        w = (torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8) * half(0)
    elif fmt == "q4_k":
        s, q = b[:, 4:16], b[:, 16:].reshape(-1, 4, 32)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        q = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        w = q * (half(0) * sc)[:, :, None] - (half(2) * mn)[:, :, None]
    else:
        lo, hi = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 1, 32)
        q = torch.stack([lo[:, :, 0] & 15, lo[:, :, 1] & 15, lo[:, :, 0] >> 4, lo[:, :, 1] >> 4], 2)
        q = (q | (torch.cat([(hi >> (2 * i)) & 3 for i in range(4)], 2) << 4)).double() - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double().reshape(-1, 2, 4, 2, 1) * half(208)[:, :, None, None, None]
        w = q.reshape(-1, 2, 4, 2, 16) * sc
    return w.reshape(rows, k)


def _host(t):
    """A GPU tensor as the host array a program uploads: bf16 as its bits."""
    return (t.view(torch.int16).cpu().numpy().view(np.uint16) if t.dtype == torch.bfloat16 else t.cpu().numpy())


# ── transformers ──

def _hf(model):
    cfg = synth_model.QWEN3_0P6B if model == "qwen3-0.6b" else synth_model.listed_shape(model)
    return dataclasses.replace(cfg, max_position_embeddings=MAX_SEQ), model == "qwen3-0.6b"


def _hf_shapes(cfg):
    """Projections of a layer as [out, in], in the order a model with types per projection lists them."""
    h, f, hd = cfg.hidden_size, cfg.intermediate_size, cfg.get_head_dim()
    q, kv = cfg.num_attention_heads * hd, cfg.kv_heads() * hd
    return {"q_proj": (q, h), "k_proj": (kv, h), "v_proj": (kv, h), "o_proj": (h, q), "gate_proj": (f, h), "up_proj": (f, h), "down_proj": (h, f)}


def _hf_fmt(fmt, layer, proj):
    if fmt != "q4_k_m":
        return fmt
    return "q6_k" if proj in ("v_proj", "down_proj") and layer % 2 == 0 else "q4_k"


def _hf_head_fmt(cfg, fmt):
    return "bf16" if fmt == "bf16" else "q6_k" if fmt != "q8_0" and cfg.hidden_size % 256 == 0 else "q8_0"


def _hf_raw(model, cfg, fmt, name):
    """(values as uploaded, their format) of one weight slot."""
    part, key = name.split("."), model + fmt + name
    if part[0] == "lm_head" or part[1] == "embed_tokens":
        shape, f = (cfg.vocab_size, cfg.hidden_size), _hf_head_fmt(cfg, fmt)
        key = model + fmt + "lm_head"
        head = _normal(key, shape, 0.02).bfloat16() if f == "bf16" else _blocks(key, f, *shape, 0.02)
        if part[0] == "lm_head":
            return head, f
        # the Q8_K rounding of the K-quants' activations is noise beside the stem then, also where it falls the other way
        return (_weights(head, f, shape[1]).roll(-1, 0) * (512 if fmt == "q4_k_m" else 128)).float(), "f32"
    if part[-1] == "bias":
        return _normal(key, (_hf_shapes(cfg)[part[-2]][0],), 0.5), "f32"
    if part[-2] not in _hf_shapes(cfg):
        return _normal(key, (cfg.get_head_dim() if part[-2] in ("q_norm", "k_norm") else cfg.hidden_size,), 0.1, 1.0), "f32"
    (n, k), f = _hf_shapes(cfg)[part[-2]], _hf_fmt(fmt, int(part[2]), part[-2])
    return (_normal(key, (n, k), 0.02).bfloat16() if f == "bf16" else _blocks(key, f, n, k, 0.02)), f


def _load_hf(ctx, model, fmt):
    cfg, qk_norm = _hf(model)
    types = None
    if fmt == "q4_k_m":
        types = [CODE[_hf_fmt(fmt, i, p)] for i in range(cfg.num_hidden_layers) for p in _hf_shapes(cfg)]
    m = HfModel(ctx, cfg, CODE.get(fmt, DTYPE_Q8_0), qk_norm, proj_dtypes=types)
    for i, (name, *_) in enumerate(m.weight_slots()):
        raw, f = _hf_raw(model, cfg, fmt, name)
        if name == "lm_head.weight" and f != "bf16":
            m.set_lm_head_blocks(CODE[f], _host(raw))
        else:
            (m.set_weight_nk if f == "bf16" else m.set_weight)(i, _host(raw))
    m.finalize(MAX_SEQ)
    return m


def _rms(x, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _softmax_rows(q, k, v, scale, seen):
    """q [H, T, d] over k, v [H, T, d]; seen(i, j): which keys j a query i sees. Queries a few hundred at a time."""
    out, j = [], torch.arange(k.shape[1], device="cuda")
    for at in range(0, q.shape[1], 512):
        i = torch.arange(at, min(at + 512, q.shape[1]), device="cuda")
        s = (q[:, i] @ k.transpose(1, 2)) * scale
        out.append(s.masked_fill(~seen(i[:, None], j[None, :]), -math.inf).softmax(-1) @ v)
    return torch.cat(out, 1)


def _rotate(x, base, dims):
    """Pairs (i, i + dims / 2) of the first `dims` of the last axis of [T, ..., d] turned by t * base^(-2i / dims)."""
    f = base ** (-torch.arange(0, dims, 2, device="cuda", dtype=torch.float64) / dims)
    a = (torch.arange(x.shape[0], device="cuda", dtype=torch.float64)[:, None] * f).reshape((-1,) + (1,) * (x.dim() - 2) + (dims // 2,))
    lo, hi = x[..., :dims // 2], x[..., dims // 2:dims]
    return torch.cat([lo * a.cos() - hi * a.sin(), hi * a.cos() + lo * a.sin(), x[..., dims:]], -1)


def _exact_hf(model, fmt, ids):
    """Logits of the last of `ids`; K and V rows rounded to bf16, as the cache holds them."""
    cfg, qk_norm = _hf(model)
    eps, hd, heads, kvh = cfg.rms_norm_eps, cfg.get_head_dim(), cfg.num_attention_heads, cfg.kv_heads()

    def get(name):
        raw, f = _hf_raw(model, cfg, fmt, name)
        part = name.split(".")[-2]
        return raw.double() if f in ("f32", "bf16") else _weights(raw, f, _hf_shapes(cfg)[part][1] if part in _hf_shapes(cfg) else cfg.hidden_size)
    x, T = get("model.embed_tokens.weight")[ids], len(ids)
    for i in range(cfg.num_hidden_layers):
        p = f"model.layers.{i}."
        h = _rms(x, eps) * get(p + "input_layernorm.weight")
        q, k, v = (h @ get(p + f"self_attn.{n}_proj.weight").T + (get(p + f"self_attn.{n}_proj.bias") if cfg.attention_bias else 0) for n in "qkv")
        q, k, v = q.view(T, heads, hd), k.view(T, kvh, hd), v.view(T, kvh, hd)
        if qk_norm:
            q, k = _rms(q, eps) * get(p + "self_attn.q_norm.weight"), _rms(k, eps) * get(p + "self_attn.k_norm.weight")
        q, k = _rotate(q, cfg.rope_theta, hd), _rotate(k, cfg.rope_theta, hd)
        k, v = (t.bfloat16().double().repeat_interleave(heads // kvh, 1).transpose(0, 1) for t in (k, v))
        a = _softmax_rows(q.transpose(0, 1), k, v, hd ** -0.5, lambda i, j: j <= i)
        x = x + a.transpose(0, 1).reshape(T, heads * hd) @ get(p + "self_attn.o_proj.weight").T
        h = _rms(x, eps) * get(p + "post_attention_layernorm.weight")
        h = torch.nn.functional.silu(h @ get(p + "mlp.gate_proj.weight").T) * (h @ get(p + "mlp.up_proj.weight").T)
        x = x + h @ get(p + "mlp.down_proj.weight").T
    return (_rms(x[-1:], eps) * get("model.norm.weight")) @ get("lm_head.weight").T


# ── list-of-layers decoders ──

def _block_cfg(model):
    family, size = model.split("-")
    return {"nokuvik": synth_model.nokuvik_shape, "ludalix": synth_model.ludalix_shape}[family](size)


def _block_shapes(cfg):
    """{name: shape} of every tensor, matrices [out, in]."""
    w, out = cfg["width"], {}
    pre = cfg["architecture"] == "Nokuvik"

    def put(prefix, **shapes):
        out.update({prefix + k.replace("_", "."): s for k, s in shapes.items()})
    put("", embed=(cfg["vocab"], w), head=(cfg["vocab"], w), final_norm=(w,))
    for i, layer in enumerate(cfg["layers"]):
        p, m, mlp = f"l{i}.", layer["mixer"], layer.get("mlp")
        for n in ("norm1", "norm2")[:2 if mlp else 1]:
            put(p, **{n: (w,)}, **({n + "b": (w,)} if pre else {}))
        p += "mix."
        if layer["type"] == "latent_attention":
            h, d, r, vd, qr, kr = (m[k] for k in ("heads", "dim", "rot_dim", "vdim", "q_rank", "kv_rank"))
            put(p, dq=(qr, w), dq_norm=(qr,), uq=(h * (d + r), qr), dkv=(kr + r, w), dkv_norm=(kr,), uk=(h * d, kr), uv=(h * vd, kr),
                g=(h * vd, w), o=(w, h * vd))
        elif layer["type"] == "mamba1":
            n, s, r = m["inner"], m["state"], m["dt_rank"]
            out.update({p + "in": (2 * n, w), p + "A_log": (n, s)})
            put(p, conv=(n, m["conv"]), conv_b=(n,), x=(r + 2 * s, n), dt=(n, r), dt_b=(n,), D=(n,), o=(w, n))
        elif layer["type"] == "rglru":
            n, b = m["width"], m["blocks"]
            put(p, y=(n, w), y_b=(n,), x=(n, w), x_b=(n,), conv=(n, m["conv"]), conv_b=(n,), ra=(n, n // b), ra_b=(n,), ri=(n, n // b),
                ri_b=(n,), lam=(n,), o=(w, n))
        elif layer["type"] == "attention":
            h, g, d, vd = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
            put(p, q=(h * d, w), q_norm=(d,), o=(w, h * vd))
            if m.get("kv_from") is None:
                put(p, k=(g * d, w), v=(g * vd, w), k_norm=(d,))
        else:
            h, d, vd = m["heads"], m["dim"], m["vdim"]
            put(p, q=(h * d, w), k=(h * d, w), v=(h * vd, w), g=(h * vd, w), i=(h, w), i_b=(h,), f=(h, w), f_b=(h,), norm=(h * vd,), o=(w, h * vd))
        p = f"l{i}.mlp."
        if mlp and mlp["kind"] == "dense":
            put(p, gate=(mlp["ff"], w), up=(mlp["ff"], w), down=(w, mlp["ff"]))
        elif mlp:
            put(p, router=(mlp["router"]["experts"], w))
            for e in range(mlp["router"]["experts"]):
                put(f"{p}e{e}.", gate=(mlp["expert"]["ff"], w), up=(mlp["expert"]["ff"], w), down=(w, mlp["expert"]["ff"]))
    return out


def _block_raw(model, shapes, name):
    shape, leaf, key = shapes[name], name.split(".")[-1], model + name
    if name == "embed":  # a stem well above what the layers add to it: which experts a token takes does not hang on rounding
        return _block_raw(model, shapes, "head").float().roll(-1, 0) * (256 if model.startswith("nokuvik") else 1024)
    if "norm" in leaf:
        return _normal(key, shape, 0.1, 1.0)
    if leaf == "A_log":
        return _normal(key, shape, 0.1) + torch.arange(1, shape[1] + 1, device="cuda").log()
    if name.endswith("dt.b") or leaf == "lam":
        return _normal(key, shape, 1.0, -2.0 if leaf == "lam" else -4.0)
    if leaf in ("b", "conv"):
        return _normal(key, shape, 0.3)
    if len(shape) == 1:
        return _normal(key, shape, 1.0)
    # no norm stands ahead of Ludalix's layers: what reads the residual is sized for it
    reads = model.startswith("ludalix") and leaf in ("q", "k", "v", "g", "i", "f", "router", "gate", "up")
    return _normal(key, shape, shape[1] ** -0.5 / (16 if reads else 1)).bfloat16()


def _load_block(ctx, model):
    cfg = _block_cfg(model)
    m, shapes = BlockModel(ctx, cfg, DTYPE_BF16), _block_shapes(cfg)
    for i, (name, *_) in enumerate(m.weight_slots()):
        m.set_weight_nk(i, _host(_block_raw(model, shapes, name)))
    m.finalize(MAX_SEQ)
    return m


def _conv(x, w, b):
    return torch.nn.functional.conv1d(torch.nn.functional.pad(x.T, (w.shape[1] - 1, 0))[None], w[:, None], b, groups=len(w))[0].T


def _latent_attention(h, m, t, eps):
    T, H, d, r = len(h), m["heads"], m["dim"], m["rot_dim"]
    q = (_rms(h @ t["dq"].T, eps) * t["dq.norm"] @ t["uq"].T).view(T, H, d + r)
    down = h @ t["dkv"].T
    c = _rms(down[:, :m["kv_rank"]], eps) * t["dkv.norm"]
    kr = _rotate(down[:, m["kv_rank"]:], m["rot"]["base"], m["rot"]["dims"])
    q = torch.cat([q[..., :d], _rotate(q[..., d:], m["rot"]["base"], m["rot"]["dims"])], -1)
    k = torch.cat([(c @ t["uk"].T).view(T, H, d), kr[:, None].expand(T, H, r)], -1)
    v = (c @ t["uv"].T).view(T, H, m["vdim"])
    a = _softmax_rows(q.transpose(0, 1), k.transpose(0, 1), v.transpose(0, 1), m["scale"], lambda i, j: (j <= i) & (i - j < m["mask"]["size"]))
    return (a.transpose(0, 1).reshape(T, -1) * (h @ t["g"].T).sigmoid()) @ t["o"].T


def _mamba1(h, m, t, eps):
    n, s, r = m["inner"], m["state"], m["dt_rank"]
    xz = h @ t["in"].T
    x = torch.nn.functional.silu(_conv(xz[:, :n], t["conv"], t["conv.b"]))
    p = x @ t["x"].T
    dt = torch.nn.functional.softplus(p[:, :r] @ t["dt"].T + t["dt.b"])
    A, B, C = -t["A_log"].exp(), p[:, r:r + s], p[:, r + s:]
    S, y = torch.zeros(n, s, device="cuda", dtype=torch.float64), []
    for at in range(0, len(h), 256):
        keep = (dt[at:at + 256, :, None] * A).exp()
        add = (dt * x)[at:at + 256, :, None] * B[at:at + 256, None]
        for i in range(len(keep)):
            S = torch.addcmul(add[i], keep[i], S)
            add[i] = S
        y.append((add @ C[at:at + 256, :, None])[..., 0])
    return ((torch.cat(y) + t["D"] * x) * torch.nn.functional.silu(xz[:, n:])) @ t["o"].T


def _rglru(h, m, t, eps):
    b = m["blocks"]
    y = torch.nn.functional.gelu(h @ t["y"].T + t["y.b"], approximate="tanh")
    u = _conv(h @ t["x"].T + t["x.b"], t["conv"], t["conv.b"])

    def gate(name):
        w = t[name].view(b, -1, t[name].shape[1])
        return (torch.einsum("tbi,boi->tbo", u.view(len(u), b, -1), w).reshape(u.shape) + t[name + ".b"]).sigmoid()
    log_a = -8.0 * gate("ra") * torch.nn.functional.softplus(t["lam"])
    keep, S = log_a.exp(), (-(2 * log_a).expm1()).sqrt() * gate("ri") * u
    for i in range(1, len(h)):
        S[i] += keep[i] * S[i - 1]
    return (S * y) @ t["o"].T


def _mlstm(h, m, t, eps):
    T, H, d = len(h), m["heads"], m["dim"]
    q, k, v = ((h @ t[n].T).view(T, H, -1).transpose(0, 1) for n in "qkv")
    i, f = (m["gate_cap"] * torch.tanh((h @ t[n].T + t[n + ".b"]) / m["gate_cap"]) for n in "if")
    F = torch.nn.functional.logsigmoid(f).cumsum(0).T
    lw = (F[:, :, None] - F[:, None] + i.T[:, None]).masked_fill(torch.ones(T, T, device="cuda").triu(1).bool(), -math.inf)
    top = torch.maximum(lw.amax(-1), F)
    s = (lw - top[..., None]).exp() * (q @ k.transpose(1, 2)) * d ** -0.5
    o = (s @ v) / (torch.maximum(s.sum(-1).abs(), (-top).exp()) + 1e-6)[..., None]
    return (_rms(o, eps).transpose(0, 1).reshape(T, -1) * t["norm"] * (h @ t["g"].T).sigmoid()) @ t["o"].T


def _window_attention(h, m, t, eps, keys, i):
    T, H, G = len(h), m["heads"], m["kv_heads"]
    if m.get("kv_from") is None:
        keys[i] = (_rms((h @ t["k"].T).view(T, G, -1), eps) * t["k.norm"], (h @ t["v"].T).view(T, G, -1))
    k, v = (x.repeat_interleave(H // G, 1).transpose(0, 1) for x in keys[i if m.get("kv_from") is None else m["kv_from"]])
    q = (_rms((h @ t["q"].T).view(T, H, -1), eps) * t["q.norm"]).transpose(0, 1)
    a = _softmax_rows(q, k, v, m["scale"], lambda i, j: (j <= i) & ((i - j < m["mask"]["size"]) | (j < m["mask"]["keep_first"])))
    return a.transpose(0, 1).reshape(T, -1) @ t["o"].T


def _feed_forward(h, mlp, t):
    silu = torch.nn.functional.silu
    if "limit" in mlp:
        g, u = (h @ t("gate").T).clamp(max=mlp["limit"]), (h @ t("up").T).clamp(-mlp["limit"], mlp["limit"])
        return (g * (1.702 * g).sigmoid() * (u + 1)) @ t("down").T
    if mlp["kind"] == "dense":
        return (silu(h @ t("gate").T) * (h @ t("up").T)) @ t("down").T
    weight, chosen = (h @ t("router").T).sigmoid().topk(mlp["router"]["top"], 1)
    y = torch.zeros_like(h)
    for e in range(mlp["router"]["experts"]):
        rows, place = (chosen == e).nonzero(as_tuple=True)
        z = weight[rows, place][:, None] * h[rows]
        y[rows] += (silu(z @ t(f"e{e}.gate").T) * (z @ t(f"e{e}.up").T)) @ t(f"e{e}.down").T
    return y


def _exact_block(model, ids):
    cfg = _block_cfg(model)
    eps, shapes, pre, mu = cfg["norm"]["eps"], _block_shapes(cfg), cfg["architecture"] == "Nokuvik", cfg.get("residual_mult", 1.0)

    def get(name):
        return _block_raw(model, shapes, name).double()
    x, keys, width = get("embed")[ids] * cfg["embedding"]["scale"], {}, cfg["width"]
    if not pre:
        c = torch.arange(width, device="cuda", dtype=torch.float64)
        a = torch.arange(len(ids), device="cuda", dtype=torch.float64)[:, None] * 10000.0 ** (-(c - c % 2) / width)
        x = x + torch.where(c % 2 == 0, a.sin(), a.cos())
    mixers = {"latent_attention": _latent_attention, "mamba1": _mamba1, "rglru": _rglru, "mlstm": _mlstm}
    for i, layer in enumerate(cfg["layers"]):
        p = f"l{i}."
        t = {n[len(p) + 4:]: get(n) for n in shapes if n.startswith(p + "mix.")}
        h = _rms(x, eps) * get(p + "norm1") if pre else x
        y = _window_attention(h, layer["mixer"], t, eps, keys, i) if layer["type"] == "attention" else mixers[layer["type"]](h, layer["mixer"], t, eps)
        x = x + mu * _rms(y, eps) * get(p + ("norm1b" if pre else "norm1"))
        if layer.get("mlp"):
            h = _rms(x, eps) * get(p + "norm2") if pre else x
            y = _feed_forward(h, layer["mlp"], lambda n: get(p + "mlp." + n))
            x = x + mu * _rms(y, eps) * get(p + ("norm2b" if pre else "norm2"))
    return (_rms(x[-1:], eps) * get("final.norm")) @ get("head").T


# ── preparing and running ──

_CTX, _MODELS = [], {}


def _context():
    if not _CTX:
        _CTX.append(Context(0))
    return _CTX[0]


def _model(model, fmt):
    if (model, fmt) not in _MODELS:
        ctx = _context()
        _MODELS[model, fmt] = _load_block(ctx, model) if model.startswith(("nokuvik", "ludalix")) else _load_hf(ctx, model, fmt)
    return _MODELS[model, fmt]


class _Ptr:
    """A tensor as the argument of a kernel-level entry point."""

    def __init__(self, t):
        self.t, self.ptr = t, ctypes.c_void_p(t.data_ptr())


def _prompt(case, seed):
    vocab = _block_cfg(case["model"])["vocab"] if case["model"].startswith(("nokuvik", "ludalix")) else _hf(case["model"])[0].vocab_size
    return np.random.RandomState(seed % (1 << 32)).randint(0, vocab, case["prompt"]).astype(np.int64), vocab


def _operands(case, seed):
    g = torch.Generator("cuda").manual_seed(seed)

    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda")
    if case["op"] == "gemv":
        k, n = case["k"], case["n"]
        w = normal(n, k).mul_(0.02).bfloat16() if case["fmt"] == "bf16" else _blocks(f"{seed}", case["fmt"], n, k, 0.02)
        return normal(1, k), w
    if case["op"] == "gemm":
        m, k, n = case["m"], case["k"], case["n"]
        return normal(m, k).bfloat16(), normal(*((n, k) if case["nk"] else (k, n))).mul_(0.02).bfloat16()
    b, h, kvh, hd, rows = (case[x] for x in ("b", "h", "kvh", "hd", "len"))
    return normal(b, h, hd), normal(b, kvh, rows, hd).bfloat16(), normal(b, kvh, rows, hd).bfloat16()


def prepare(case, seed):
    if case["op"] in ("reply", "prompt"):
        return {"case": case, "model": _model(case["model"], case["fmt"]), "ids": _prompt(case, seed)[0], "seed": seed}
    t = _operands(case, seed)
    shape = {"gemv": lambda: (1, case["n"]), "gemm": lambda: (case["m"], case["n"]), "attention": lambda: (case["b"], case["h"] * case["hd"])}[case["op"]]()
    out = torch.zeros(shape, device="cuda")
    return {"case": case, "ctx": _context(), "args": [_Ptr(x) for x in t], "out": out, "out_arg": _Ptr(out)}


def run(state):
    case = state["case"]
    if case["op"] == "reply":
        m = state["model"]
        m.reset_kv_cache()
        tokens = m.generate(state["ids"], case["new"], DEFAULT if case["sampled"] else GREEDY, seed=state["seed"] & 0xFFFF)
        return {"tokens": tokens, "logits": m.run_kv(tokens[-1:])}
    if case["op"] == "prompt":
        m = state["model"]
        m.reset_kv_cache()
        if case["prompt"] > 1:
            m.prefill(state["ids"][:-1], want_logits=False)
        return m.run_kv(state["ids"][-1:])
    ctx, a, out = state["ctx"], state["args"], state["out_arg"]
    if case["op"] == "gemv":
        {"bf16": ctx.gemv_bf16_nk, "q8_0": ctx.gemv_q8_0, "q4_0": ctx.gemv_q4_0, "q4_k": ctx.gemv_q4_k, "q6_k": ctx.gemv_q6_k}[case["fmt"]](
            *a, out, 1, case["k"], case["n"])
    elif case["op"] == "gemm":
        (ctx.gemm_bf16_nk if case["nk"] else ctx.gemm_bf16)(*a, out, case["m"], case["k"], case["n"])
    else:
        ctx.gqa_decode_attn(*a, out, case["b"], case["h"], case["kvh"], case["hd"], case["len"], case["len"], case["hd"] ** -0.5)
    return state["out"]


def exact(case, seed):
    with torch.no_grad():
        if case["op"] in ("reply", "prompt"):
            ids, vocab = _prompt(case, seed)
            walk = (ids[-1] + 1 + np.arange(case.get("new", 0))) % vocab  # the lead of every next token
            ids = torch.from_numpy(np.concatenate([ids, walk])).cuda()
            logits = _exact_block(case["model"], ids) if case["model"].startswith(("nokuvik", "ludalix")) else _exact_hf(case["model"], case["fmt"], ids)
            return logits if case["op"] == "prompt" else {"tokens": None, "logits": logits}
        t = _operands(case, seed)
        if case["op"] == "gemv":
            return t[0].double() @ _weights(t[1], case["fmt"], case["k"]).T
        if case["op"] == "gemm":
            return t[0].double() @ (t[1].double().T if case["nk"] else t[1].double())
        q, k, v = (x.double() for x in t)
        k, v = (x.repeat_interleave(case["h"] // case["kvh"], 1) for x in (k, v))
        p = ((k @ q[..., None])[..., 0] * case["hd"] ** -0.5).softmax(-1)
        return (p[:, :, None] @ v)[:, :, 0].reshape(case["b"], -1)


# ── what a pass cannot do without ──

def _per_weight(fmt):
    return 2.0 if fmt == "bf16" else BLOCK[fmt][1] / BLOCK[fmt][0]


def work(case):
    if case["op"] == "gemv":
        return {"bytes": case["n"] * case["k"] * _per_weight(case["fmt"]) + 4 * (case["n"] + case["k"]), "flops": 2 * case["n"] * case["k"]}
    if case["op"] == "gemm":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 2 * k * (m + n) + 4 * m * n, "flops": 2 * m * n * k}
    if case["op"] == "attention":
        rows = case["b"] * case["len"] * case["hd"]
        return {"bytes": 4 * rows * case["kvh"] + 8 * case["b"] * case["h"] * case["hd"], "flops": 4 * rows * case["h"]}
    P, passes = case["prompt"], case.get("new", 0) + 1  # passes over the weights behind the prompt's, logits each
    total = P - 1 + passes
    if not case["model"].startswith(("nokuvik", "ludalix")):
        cfg, _ = _hf(case["model"])
        L, h, v, hd = cfg.num_hidden_layers, cfg.hidden_size, cfg.vocab_size, cfg.get_head_dim()
        layers = [(n * k, _hf_fmt(case["fmt"], i, p)) for i in range(L) for p, (n, k) in _hf_shapes(cfg).items()]
        size, flops = sum(a * _per_weight(f) for a, f in layers), 2.0 * sum(a for a, _ in layers)
        head = v * h * _per_weight(_hf_head_fmt(cfg, case["fmt"])) + 4 * v
        row = 4 * L * cfg.kv_heads() * hd
        cache = row * (total + (P - 1) * (P > 1) + sum(P - 1 + i for i in range(1, passes + 1)))
        pairs = 4.0 * L * cfg.num_attention_heads * hd * total * total / 2
        return {"bytes": size * ((P > 1) + passes) + head * passes + cache, "flops": flops * total + pairs + 2.0 * v * h * passes}
    cfg = _block_cfg(case["model"])
    one = many = act = 0.0
    for name, s in _block_shapes(cfg).items():
        if len(s) == 2 and name != "embed":
            n = s[0] * s[1]
            share = 1.0
            if ".mlp.e" in name:
                r = cfg["layers"][int(name[1:name.index(".")])]["mlp"]["router"]
                share = r["top"] / r["experts"]
            one, act = one + 2 * n * share, act + 2 * n * share
            many += 2 * n * (share if share == 1.0 else 1 - (1 - share) ** max(P - 1, 0))
    return {"bytes": one * passes + many * (P > 1), "flops": act * total}


def tolerance(case):
    """About four times what the same tokens differ by when they go through the model another way (a prompt in two portions,
    generated tokens as a prompt); kernel-level calls: float32 sums in another order, and attention's two-piece operands."""
    if case["op"] in ("gemv", "gemm"):
        return {"rel": 3e-6, "max": 3e-5}
    if case["op"] == "attention":
        return {"rel": 1.5e-5, "max": 1e-4}
    if case["model"].startswith("nokuvik"):
        return {"rel": 8e-3, "max": 0.035, "differ": 0.0}
    if case["model"].startswith("ludalix"):
        return {"rel": 2e-3, "max": 0.01, "differ": 0.0}
    if case["fmt"] == "q4_k_m":  # activations are rounded to eight bits: sums in another order round some of them the other way
        return {"rel": 0.025, "max": 0.12, "differ": 0.0}
    return {"rel": 7e-4, "max": 4e-3, "differ": 0.0}  # rows of the cache round to bf16 the other way
