"""Performance cases: the calls a program that serves models with this framework spends its time in.

Four kinds of call, over the model shapes of the package's presets and the sizes its engines run them at:

  segment    one packed segment as the engines issue it: plan the blocks (`build_packed_arrays`), run layers
             [0, layers) over them (`packed_layers`).  Decode rows (one token per request), verify blocks (a few
             tokens per request), prefill pieces (`piece` tokens of one prompt) and mixes of them.  Returns the
             hidden states and the K / V caches the call appended to.
  prompt     a whole-prompt prefill through `LayerSkipLlama.prefill`: embedding, every layer, head; returns logits.
  attention  ragged verify / decode attention over a KV cache on its own (`_lsk.ragged_attn`), plan in hand.
  head       final norm + LM head + greedy pick (`_lsk.head_norm_argmax`); returns logits and tokens.

A case's block structure (contexts, tokens per block) follows from the case alone (`shape` seeds it); the seed of
`prepare` makes the weights, cached K / V and activations.
"""

from __future__ import annotations

import dataclasses
import math
import random

import numpy as np
import torch

DEV = "cuda"


# ----------------------------------------------------------------------------- the cases

def _segment(name, preset, layers, requests, t, ctx, max_seq, piece=0, piece_pos=0, dtype="bf16", shape=1):
    """requests blocks of t[0]..t[1] tokens at contexts ctx[0]..ctx[1]; then, with piece > 0, one block of `piece`
    prompt tokens at position piece_pos of a cache row of its own."""
    c = {"kind": "segment", "preset": preset, "dtype": dtype, "layers": layers, "requests": requests, "t_lo": t[0],
         "t_hi": t[1], "ctx_lo": ctx[0], "ctx_hi": ctx[1], "piece": piece, "piece_pos": piece_pos,
         "max_seq": max_seq, "shape": shape}
    return {"name": name, **c} if name else c


def listed() -> list:
    return [
        # single-stream interactive decoding: one request's next draft token through a 1B shape's shallow layers;
        # every launch is at its floor
        _segment("decode_1b_b1", "llama3.2-1b", 6, 1, (1, 1), (300, 400), 2048),
        # the decode batch of an 8B server: 32 requests, one token each, contexts up to prompt 1024 + 256 new tokens
        _segment("decode_8b_b32", "llama3-8b", 2, 32, (1, 1), (128, 1280), 2048),
        # its usual verification step: about ten of the requests check their drafts (3 to 9 tokens each)
        _segment("verify_8b_b10", "llama3-8b", 2, 10, (3, 9), (128, 1280), 2048),
        # synchronous speculation on the 1B shape: all 64 requests verify 6 drafts + 1 (448 rows)
        _segment("verify_1b_b64", "llama3.2-1b", 2, 64, (7, 7), (512, 768), 1024),
        # piggybacked prefill on an MHA model: 32 decoding requests and a 256-token piece of a waiting prompt
        _segment("piece_7b_b32", "llama2-7b", 2, 32, (1, 1), (256, 1100), 1280, piece=256, piece_pos=256),
        # a separate prefill's piece (512 tokens is the engines' default), the second of its prompt
        _segment("prefill_8b_512", "llama3-8b", 2, 0, (1, 1), (1, 1), 2048, piece=512, piece_pos=512),
        # a long prompt in one call, odd length, near the 8B shape's position limit
        _segment("prefill_8b_4001", "llama3-8b", 2, 0, (1, 1), (1, 1), 8192, piece=4001, piece_pos=0),
        # a whole model call: prompt in, logits out (1B shape, every layer, the 128256-row head)
        {"name": "prompt_1b_1517", "kind": "prompt", "preset": "llama3.2-1b", "layers": 16, "tokens": 1517,
         "max_seq": 2048},
        # verify attention of a large batch: 256 requests, contexts of median 1500 up to 8192, 1 to 9 rows each
        {"name": "attention_8b_b256", "kind": "attention", "preset": "llama3-8b", "requests": 256,
         "ctx_median": 1500, "ctx_max": 8183, "t_lo": 1, "t_hi": 9, "shape": 1},
        # the head over the rows of a step (drafts and verify tokens share one launch)
        {"name": "head_8b_32", "kind": "head", "preset": "llama3-8b", "rows": 32},
        # the fp32 model (the token-identity configuration): 4 requests verify 4 drafts + 1
        _segment("verify_1b_fp32_b4", "llama3.2-1b", 2, 4, (5, 5), (16, 192), 256, dtype="fp32"),
        # and prefills a prompt of its length range
        _segment("prefill_1b_fp32_121", "llama3.2-1b", 2, 0, (1, 1), (1, 1), 256, piece=121, dtype="fp32"),
    ]


def _log(rng, lo, hi) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["decode", "verify", "mixed", "piece", "piece", "prompt", "attention", "head", "fp32"])
    preset = rng.choice(["llama3-8b", "llama3-8b", "llama3.2-1b", "llama2-7b"])
    shape = rng.randrange(1, 1 << 20)
    if kind in ("decode", "verify", "mixed"):
        b = _log(rng, 1, 128 if kind == "decode" else 64)
        hi = _log(rng, 64, 1900)
        t = (1, 1) if kind != "verify" else (rng.randint(1, 3), rng.randint(3, 9))
        piece = _log(rng, 16, 512) if kind == "mixed" else 0
        return _segment(None, preset, rng.randint(1, 2), b, t, (rng.randint(1, 64), hi), 2048, piece=piece,
                        piece_pos=rng.randint(0, 1024) if piece else 0, shape=shape)
    if kind == "piece":
        n = _log(rng, 64, 4096 if preset != "llama2-7b" else 2048)
        return _segment(None, preset, 1, 0, (1, 1), (1, 1), 8192, piece=n,
                        piece_pos=rng.choice([0, rng.randint(0, 2048)]), shape=shape)
    if kind == "prompt":
        return {"kind": "prompt", "preset": "llama3.2-1b", "layers": rng.randint(2, 16), "tokens": _log(rng, 16, 2048),
                "max_seq": 2048}
    if kind == "attention":
        med = _log(rng, 200, 3000)
        return {"kind": "attention", "preset": preset, "requests": _log(rng, 4, 256 if preset != "llama2-7b" else 64),
                "ctx_median": med, "ctx_max": 8183, "t_lo": 1, "t_hi": rng.randint(1, 9), "shape": shape}
    if kind == "head":
        return {"kind": "head", "preset": preset, "rows": _log(rng, 1, 512)}
    if rng.random() < 0.5:
        return _segment(None, "llama3.2-1b", rng.randint(1, 2), _log(rng, 1, 16), (1, rng.randint(1, 9)),
                        (rng.randint(1, 16), _log(rng, 32, 230)), 256, dtype="fp32", shape=shape)
    return _segment(None, "llama3.2-1b", 1, 0, (1, 1), (1, 1), 256, piece=_log(rng, 9, 200), dtype="fp32", shape=shape)


# ----------------------------------------------------------------------------- what a case consists of

def _cfg(case):
    from thesis_amd.common.model import PRESETS

    return dataclasses.replace(PRESETS[case["preset"]], **({"n_layers": case["layers"]} if "layers" in case else {}))


def _dtype(case):
    return torch.float32 if case.get("dtype") == "fp32" else torch.bfloat16


def _blocks(case):
    """(rows, pos0, T) of a segment's blocks in packed order (T ascending, then row)."""
    r = random.Random(case["shape"])
    b = [(i, r.randint(case["ctx_lo"], max(case["ctx_lo"], case["ctx_hi"])), r.randint(case["t_lo"], case["t_hi"]))
         for i in range(case["requests"])]
    if case["piece"]:
        b.append((case["requests"], case["piece_pos"], case["piece"]))
    b.sort(key=lambda x: (x[2], x[0]))
    return tuple(np.array([x[j] for x in b], dtype=np.int64) for j in range(3))


def _contexts(case):
    """(contexts, tokens per request) of an attention case: lognormal contexts."""
    r = random.Random(case["shape"])
    ctx = [min(case["ctx_max"], max(64, int(r.lognormvariate(math.log(case["ctx_median"]), 0.5))))
           for _ in range(case["requests"])]
    t = [r.randint(case["t_lo"], case["t_hi"]) for _ in ctx]
    return np.array(ctx, dtype=np.int64), np.array(t, dtype=np.int64)


def _gen(seed, part):
    return torch.Generator(device=DEV).manual_seed((int(seed) * 1000003 + part) % (1 << 62))


def _normal(gen, *shape, dtype=torch.bfloat16, std=1.0):
    return torch.empty(*shape, dtype=dtype, device=DEV).normal_(0.0, std, generator=gen)


def _layer(cfg, seed, i, dtype):
    """Layer i's [out, in] weights at the usual N(0, 0.02) initialisation, norms around 1."""
    g = _gen(seed, 10 + i)
    qd, kvd = cfg.n_heads * cfg.head_dim, cfg.n_kv_heads * cfg.head_dim

    def mat(r, c):
        return _normal(g, r, c, dtype=dtype, std=0.02)

    def gain():
        return _normal(g, cfg.dim, dtype=dtype, std=0.1).add_(1.0)

    return [mat(qd + 2 * kvd, cfg.dim), mat(cfg.dim, qd), mat(2 * cfg.intermediate_size, cfg.dim),
            mat(cfg.dim, cfg.intermediate_size), gain(), gain()]


def _prefix(cfg, seed, i, rows, pos0, n_rows, max_seq, dtype):
    """Layer i's cached K and V [n_rows, Hkv, max_seq, D]: N(0, 1) at each row's first pos0 positions, zero after."""
    g = _gen(seed, 5000 + i)
    lens = torch.zeros(n_rows, dtype=torch.long, device=DEV)
    if len(rows):
        lens[torch.from_numpy(rows).to(DEV)] = torch.from_numpy(pos0).to(DEV)
    keep = (torch.arange(max_seq, device=DEV)[None] < lens[:, None])[:, None, :, None]
    out = []
    for _ in range(2):
        x = _normal(g, n_rows, cfg.n_kv_heads, max_seq, cfg.head_dim, dtype=dtype)
        out.append(x.mul_(keep))
    return out


def _embedding(cfg, seed, part):
    return _normal(_gen(seed, part), cfg.vocab_size, cfg.dim, std=0.02)


def _model(cfg, seed, dtype, max_seq, embed=None, lm_head=None, norm=None):
    from thesis_amd import _lsk
    from thesis_amd.common.model import LayerSkipLlama, LayerWeights

    heads = (cfg.n_heads, cfg.n_kv_heads, cfg.head_dim)
    layers = [LayerWeights.from_dense(*_layer(cfg, seed, i, dtype), heads) for i in range(cfg.n_layers)]
    head = _lsk.as_gemm_weight(lm_head) if lm_head is not None else None
    return LayerSkipLlama(cfg, embed, layers, norm, head, DEV, dtype, max_seq)


def _n_rows(case):
    return case["requests"] + (1 if case["piece"] else 0)


def prepare(case: dict, seed: int):
    from thesis_amd import _lsk

    cfg, dtype = _cfg(case), _dtype(case)
    if case["kind"] == "segment":
        rows, pos0, T = _blocks(case)
        m = _model(cfg, seed, dtype, case["max_seq"])
        m.allocate_cache(_n_rows(case), case["max_seq"])
        for i in range(cfg.n_layers):
            k, v = _prefix(cfg, seed, i, rows, pos0, _n_rows(case), case["max_seq"], dtype)
            m.cache.kstore[i].copy_(_lsk.k_to_frag(k) if m.cache.frag_k else k)
            m.cache.vb[i].copy_(_lsk.v_to_blocked(v))
            del k, v
        x = _normal(_gen(seed, 1), int(T.sum()), cfg.dim, dtype=dtype)
        return {"kind": "segment", "model": m, "blocks": (rows, pos0, T), "x": x}
    if case["kind"] == "prompt":
        m = _model(cfg, seed, dtype, case["max_seq"], _embedding(cfg, seed, 2), _embedding(cfg, seed, 3),
                   _normal(_gen(seed, 4), cfg.dim, std=0.1).add_(1.0))
        m.allocate_cache(1, case["max_seq"])
        return {"kind": "prompt", "model": m, "tokens": _prompt(case, cfg, seed)}
    if case["kind"] == "attention":
        ctx, T = _contexts(case)
        q, k, v = _attention_inputs(case, cfg, seed)
        blocks = np.stack([np.cumsum(T) - T, ctx, T, np.arange(len(T))], axis=1).astype(np.int32)
        G, Hkv, D = cfg.n_heads // cfg.n_kv_heads, cfg.n_kv_heads, cfg.head_dim
        # the split a cache of this size uses (KVCache)
        split = _lsk.ATTN_SPLIT if len(T) * Hkv >= 1024 else 2048
        slots = _lsk.cu_count(DEV)
        cap = _lsk.attn_rows_cap(blocks, G, split, Hkv, D, slots)
        works, groups, n_parts = _lsk.attn_plan(blocks, G, split, cap)
        recs, n_rounds = _lsk.attn_schedule(works, Hkv, slots)

        def up(a):
            return torch.from_numpy(a).to(DEV)

        return {"kind": "attention", "q": q, "k": k, "v": v, "blocks": up(blocks), "works": up(works),
                "n_works": len(works), "groups": up(groups) if len(groups) else None, "n_groups": len(groups),
                "n_parts": n_parts, "out": torch.empty(q.shape[0], cfg.n_heads * D, dtype=dtype, device=DEV),
                "n_heads": cfg.n_heads, "scale": 1.0 / math.sqrt(D), "recs": up(recs), "n_rounds": n_rounds,
                "slots": slots, "cap": cap,
                "ws": torch.empty(max(_lsk.attn_workspace_bytes(n_parts, Hkv, D), 1), dtype=torch.uint8, device=DEV)}
    w = _lsk.PackedWeight(_embedding(cfg, seed, 3))
    n = case["rows"]
    return {"kind": "head", "w": w, "norm": _normal(_gen(seed, 4), cfg.dim, std=0.1).add_(1.0), "eps": cfg.norm_eps,
            "h": _normal(_gen(seed, 1), n, cfg.dim),
            "ids": torch.empty(n, dtype=torch.long, device=DEV),
            "logits": torch.empty(n, cfg.vocab_size, dtype=dtype, device=DEV),
            "ws": torch.empty(int(_lsk.load().lsk_head_norm_workspace_bytes(n, cfg.vocab_size, cfg.dim)),
                              dtype=torch.uint8, device=DEV)}


def _prompt(case, cfg, seed) -> list:
    r = random.Random(int(seed) * 7 + 1)
    return [r.randrange(cfg.vocab_size) for _ in range(case["tokens"])]


def _attention_inputs(case, cfg, seed):
    """q [N, Hq, D], and K / V in the cache's storage layouts, N(0, 1)."""
    ctx, T = _contexts(case)
    S = (int((ctx + T).max()) + 63) // 64 * 64
    B, Hkv, D = len(T), cfg.n_kv_heads, cfg.head_dim
    g = _gen(seed, 6)
    return (_normal(g, int(T.sum()), cfg.n_heads, D), _normal(g, B, Hkv, S // 32, D // 16, 64, 8),
            _normal(g, B, Hkv, S // 32, D, 32))


@torch.inference_mode()
def run(state):
    from thesis_amd import _lsk
    from thesis_amd.solutions.packed import build_packed_arrays, packed_layers

    s = state
    if s["kind"] == "segment":
        m = s["model"]
        pb = build_packed_arrays(m, *s["blocks"])
        h = packed_layers(m, s["x"], pb, 0, m.n_layers)
        return {"hidden": h, "k": m.cache.kstore, "v": m.cache.vb}
    if s["kind"] == "prompt":
        m = s["model"]
        logits, _ = m.prefill(s["tokens"], 0)
        return {"logits": logits, "k": m.cache.kstore, "v": m.cache.vb}
    if s["kind"] == "attention":
        _lsk.ragged_attn(s["q"], s["k"], s["v"], s["blocks"], s["works"], s["n_works"], s["groups"], s["n_groups"],
                         s["n_parts"], s["out"], s["n_heads"], s["scale"], s["ws"], s["recs"], s["n_rounds"],
                         s["slots"], s["cap"])
        return {"out": s["out"]}
    _lsk.head_norm_argmax(s["h"], s["norm"], s["eps"], s["w"], s["ids"], logits=s["logits"], workspace=s["ws"])
    return {"logits": s["logits"], "ids": s["ids"]}


# ----------------------------------------------------------------------------- work and tolerance

def work(case: dict) -> dict:
    cfg, es = _cfg(case), _dtype(case).itemsize
    kv = 2 * cfg.n_kv_heads * cfg.head_dim * es                       # bytes of one cached position of one layer
    if case["kind"] in ("segment", "prompt"):
        if case["kind"] == "segment":
            _, pos0, T = _blocks(case)
        else:
            pos0, T = np.array([0]), np.array([case["tokens"]])
        n, L = int(T.sum()), cfg.n_layers
        pairs = int((T * pos0 + T * (T + 1) // 2).sum())
        by = L * (cfg.layer_param_count * es + int(pos0.sum()) * kv + n * kv) + 2 * n * cfg.dim * es
        fl = L * (2.0 * n * (cfg.layer_param_count - 2 * cfg.dim) + 4.0 * cfg.n_heads * cfg.head_dim * pairs)
        if case["kind"] == "prompt":
            by += cfg.vocab_size * cfg.dim * es + cfg.vocab_size * es - n * cfg.dim * es
            fl += 2.0 * cfg.vocab_size * cfg.dim
        return {"bytes": by, "flops": fl}
    if case["kind"] == "attention":
        ctx, T = _contexts(case)
        pairs = int((T * ctx + T * (T + 1) // 2).sum())
        return {"bytes": int((ctx + T).sum()) * kv + 2 * int(T.sum()) * cfg.n_heads * cfg.head_dim * es,
                "flops": 4.0 * cfg.n_heads * cfg.head_dim * pairs}
    n = case["rows"]
    return {"bytes": (cfg.vocab_size * cfg.dim + n * cfg.dim + cfg.dim + n * cfg.vocab_size) * es + 8 * n,
            "flops": 2.0 * n * cfg.vocab_size * cfg.dim}


def tolerance(case: dict):
    """About four times the distance of these kernels to 64 bits: bf16 roundings of every operation's output over one
    or two layers (0.4 to 0.9 % of the hidden states, up to 0.8 % of the appended K / V), of a whole model call (2.8 %
    of the last layers' K / V), of the attention alone (0.21 %) and of the head (0.29 %); 32-bit sums for fp32
    (8e-7)."""
    if case.get("dtype") == "fp32":
        return {"rel": 4e-6, "max": 1e-3}
    if case["kind"] == "attention":
        return {"rel": 8e-3, "max": 0.25}
    if case["kind"] == "head":
        return {"rel": 1.2e-2, "max": 0.25, "differ": 0.01}
    return {"rel": 3e-2, "max": 0.5}


# ----------------------------------------------------------------------------- the same in 64 bits

def _rope_tables(cfg, positions):
    """cos, sin [n, D] in 64 bits (Llama 3's frequency smoothing where the configuration asks for it)."""
    d = cfg.head_dim
    inv = cfg.rope_theta ** (-torch.arange(0, d, 2, dtype=torch.float64) / d)
    s = cfg.rope_scaling
    if s:
        old, lo, hi = s["original_max_position_embeddings"], s["low_freq_factor"], s["high_freq_factor"]
        turns = old * inv / (2 * math.pi)                                # rotations over the original context
        w = ((turns - lo) / (hi - lo)).clamp(0.0, 1.0)
        inv = w * inv + (1.0 - w) * inv / s["factor"]
    ang = torch.as_tensor(positions, dtype=torch.float64)[:, None] * inv[None]
    ang = torch.cat([ang, ang], dim=1).to(DEV)
    return ang.cos(), ang.sin()


def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _rotate(x, cos, sin):
    a, b = x.chunk(2, dim=-1)
    return x * cos[:, None] + torch.cat([-b, a], dim=-1) * sin[:, None]


def _attend(q, k, v, first, scale):
    """q [T, Hq, D] at positions first.. over k, v [Hkv, >= first + T, D] -> [T, Hq, D], causal."""
    T, Hq, D = q.shape
    n, g = first + T, Hq // k.shape[0]
    out = torch.empty_like(q)
    for h in range(Hq):
        kh, vh = k[h // g, :n], v[h // g, :n]
        for a in range(0, T, 1024):
            b = min(T, a + 1024)
            s = (q[a:b, h] @ kh.T) * scale
            past = torch.arange(n, device=DEV)[None] > (first + torch.arange(a, b, device=DEV))[:, None]
            out[a:b, h] = torch.softmax(s.masked_fill(past, -math.inf), dim=-1) @ vh
    return out


def _k_layout(k, frag):
    """[B, H, S, D] -> the K cache's storage: fragments of 16 positions x 32 dims per 32-position block (bf16)."""
    if not frag:
        return k
    B, H, S, D = k.shape
    x = k.reshape(B, H, S // 32, 4, 2, 4, D // 32, 4, 8).permute(0, 1, 2, 4, 6, 7, 3, 5, 8)
    return x.reshape(B, H, S // 32, D // 16, 64, 8)


def _k_rows(kf):
    B, H, nb, nf = kf.shape[:4]
    x = kf.reshape(B, H, nb, 2, nf // 2, 4, 4, 4, 8).permute(0, 1, 2, 6, 3, 7, 4, 5, 8)
    return x.reshape(B, H, nb * 32, nf * 16)


def _v_layout(v):
    B, H, S, D = v.shape
    return v.reshape(B, H, S // 32, 32, D).transpose(-1, -2)


def _forward(cfg, seed, x, rows, pos0, T, n_rows, max_seq, dtype, layers):
    """Hidden states after `layers` layers and each layer's caches, in 64 bits."""
    off = np.concatenate([[0], np.cumsum(T)])
    positions = np.concatenate([p + np.arange(t) for p, t in zip(pos0, T)])
    cos, sin = _rope_tables(cfg, positions)
    qd, kvd, D = cfg.n_heads * cfg.head_dim, cfg.n_kv_heads * cfg.head_dim, cfg.head_dim
    ks, vs = [], []
    for i in range(layers):
        wqkv, wo, w13, w2, an, fn = _layer(cfg, seed, i, dtype)
        k, v = _prefix(cfg, seed, i, rows, pos0, n_rows, max_seq, dtype)
        k, v = k.double(), v.double()
        qkv = _rms(x, an, cfg.norm_eps) @ wqkv.double().T
        q = _rotate(qkv[:, :qd].reshape(-1, cfg.n_heads, D), cos, sin)
        kn = _rotate(qkv[:, qd:qd + kvd].reshape(-1, cfg.n_kv_heads, D), cos, sin)
        vn = qkv[:, qd + kvd:].reshape(-1, cfg.n_kv_heads, D)
        att = torch.empty_like(q)
        for j, (r, p, t) in enumerate(zip(rows.tolist(), pos0.tolist(), T.tolist())):
            a, b = int(off[j]), int(off[j + 1])
            k[r, :, p:p + t] = kn[a:b].transpose(0, 1)
            v[r, :, p:p + t] = vn[a:b].transpose(0, 1)
            att[a:b] = _attend(q[a:b], k[r], v[r], p, 1.0 / math.sqrt(D))
        x = x + att.reshape(-1, qd) @ wo.double().T
        gu = _rms(x, fn, cfg.norm_eps) @ w13.double().T
        gate, up = gu.chunk(2, dim=-1)
        x = x + (torch.nn.functional.silu(gate) * up) @ w2.double().T
        ks.append(_k_layout(k, dtype == torch.bfloat16).contiguous())
        vs.append(_v_layout(v).contiguous())
    return x, ks, vs


@torch.inference_mode()
def exact(case: dict, seed: int):
    cfg, dtype = _cfg(case), _dtype(case)
    if case["kind"] == "segment":
        rows, pos0, T = _blocks(case)
        x = _normal(_gen(seed, 1), int(T.sum()), cfg.dim, dtype=dtype).double()
        h, k, v = _forward(cfg, seed, x, rows, pos0, T, _n_rows(case), case["max_seq"], dtype, cfg.n_layers)
        return {"hidden": h, "k": k, "v": v}
    if case["kind"] == "prompt":
        ids = torch.tensor(_prompt(case, cfg, seed), dtype=torch.long, device=DEV)
        one = np.array([0], dtype=np.int64)
        h, k, v = _forward(cfg, seed, _embedding(cfg, seed, 2)[ids].double(), one, one, np.array([len(ids)]), 1,
                           case["max_seq"], dtype, cfg.n_layers)
        norm = _normal(_gen(seed, 4), cfg.dim, std=0.1).add_(1.0)
        logits = _rms(h[-1:], norm, cfg.norm_eps) @ _embedding(cfg, seed, 3).double().T
        return {"logits": logits[0], "k": k, "v": v}
    if case["kind"] == "attention":
        ctx, T = _contexts(case)
        q, kf, vb = _attention_inputs(case, cfg, seed)
        out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
        a = 0
        for r, (c, t) in enumerate(zip(ctx.tolist(), T.tolist())):
            k = _k_rows(kf[r:r + 1])[0].double()
            v = vb[r].transpose(-1, -2).reshape(cfg.n_kv_heads, -1, cfg.head_dim).double()
            out[a:a + t] = _attend(q[a:a + t].double(), k, v, c, 1.0 / math.sqrt(cfg.head_dim))
            a += t
        return {"out": out.reshape(len(out), -1)}
    h = _rms(_normal(_gen(seed, 1), case["rows"], cfg.dim).double(),
             _normal(_gen(seed, 4), cfg.dim, std=0.1).add_(1.0), cfg.norm_eps)
    w = _embedding(cfg, seed, 3)
    logits = torch.cat([h @ w[a:a + 16384].double().T for a in range(0, cfg.vocab_size, 16384)], dim=1)
    return {"logits": logits, "ids": logits.argmax(-1)}
