"""Timed cases of the paged-KV path: what a program that serves a model with this
framework asks of it, through its public entry points.

Every case is a plain dict with a ``kind``; ``listed`` names the fixed ones and
``draw`` gives others of the same kinds over the ranges below.

  gqa_decode      one query token per sequence over paged K/V
  gqa_prefill     the causal window of a prompt (or of a chunk of one) over a cache
  mla_decode      absorbed MLA, one query token per sequence, projections included
  mla_prefill     absorbed MLA over the causal window of a prompt's chunk
  dsa_decode      index scores, top-k and the sparse latent contraction
  position_free   attention over unrotated shared pages, decode to prefill windows
  spill_reload    pages to the host arena and back
  attend_spilled  a decode step over a layer part of which lies in the host arena
  decoder_prefill a prompt through a whole decoder
  decoder_decode  replayed decode steps of a whole decoder
"""

from __future__ import annotations

import math
import random

import torch

from voom_amd import ops
from voom_amd.decoder import DecoderConfig, PagedDecoder
from voom_amd.kv_paged import PagedKVCache

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
# (q heads, kv heads, head dim): SmolLM2-135M, Llama-3-8B, Qwen2.5-7B, and the
# 64-head shape of the long-context workload
HEADS = [(9, 3, 64), (32, 8, 128), (28, 4, 128), (64, 8, 128)]
THETA = 5e5
LATENT, ROPE, DN, DV = 512, 64, 128, 128
INDEX_HEADS, INDEX_DIM, TOPK = 32, 128, 2048


def listed() -> list[dict]:
    return [
        # one sequence of a small model mid-generation: a latency-bound call
        {"name": "gqa_decode_one", "kind": "gqa_decode", "batch": 1, "nq": 9, "nkv": 3, "d": 64,
         "page": 64, "ctx_min": 640, "ctx_max": 640},
        # a serving batch with contexts of all lengths: the bandwidth-bound decode step
        {"name": "gqa_decode_batch", "kind": "gqa_decode", "batch": 16, "nq": 32, "nkv": 8,
         "d": 128, "page": 64, "ctx_min": 1024, "ctx_max": 32768},
        # a chunk of a long prompt after the chunks before it (ragged sizes)
        {"name": "gqa_prefill_chunk", "kind": "gqa_prefill", "batch": 1, "nq": 32, "nkv": 8,
         "d": 128, "page": 64, "seq": 6007, "window": 2011},
        # DeepSeek/GLM decode at a serving batch
        {"name": "mla_decode_batch", "kind": "mla_decode", "batch": 8, "heads": 128, "page": 64,
         "ctx_min": 16384, "ctx_max": 16384},
        # a chunk of a prompt through absorbed MLA (ragged sizes)
        {"name": "mla_prefill_chunk", "kind": "mla_prefill", "batch": 1, "heads": 128, "page": 64,
         "seq": 4397, "window": 301},
        # one DSA step over a long context
        {"name": "dsa_decode_long", "kind": "dsa_decode", "batch": 1, "heads": 128, "page": 64,
         "seq": 131072},
        # one request over shared one-token pages, decode
        {"name": "position_free_decode", "kind": "position_free", "nq": 32, "nkv": 8, "d": 128,
         "dtype": "bf16", "keys": 32768, "queries": 1},
        # the new tokens of a request behind a shared prefix, fp16 model
        {"name": "position_free_window", "kind": "position_free", "nq": 28, "nkv": 4, "d": 128,
         "dtype": "f16", "keys": 8003, "queries": 250},
        # an idle request's cache leaves the device and comes back
        {"name": "spill_reload", "kind": "spill_reload", "layers": 2, "pages": 256, "page": 64,
         "nkv": 8, "d": 128},
        # a decode step of a request whose cache exceeds its device budget
        {"name": "attend_spilled", "kind": "attend_spilled", "nq": 64, "nkv": 8, "d": 128,
         "page": 64, "seq": 32801, "spilled": 200},
        # time to first token of a whole model
        {"name": "decoder_prefill", "kind": "decoder_prefill", "tokens": 512},
        # token after token of a whole model
        {"name": "decoder_decode", "kind": "decoder_decode", "prompt": 512, "steps": 16},
    ]


def _log(rng: random.Random, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random) -> dict:
    """One more case of the ranges that the listed ones stand for."""
    kind = rng.choice(["gqa_decode", "gqa_decode", "gqa_prefill", "gqa_prefill", "mla_decode",
                       "mla_prefill", "dsa_decode", "position_free", "position_free",
                       "spill_reload", "attend_spilled", "decoder_prefill", "decoder_decode"])
    if kind == "gqa_decode":
        nq, nkv, d = rng.choice(HEADS)
        batch = _log(rng, 1, 64)
        hi = _log(rng, 48, min(131072, 266000 // batch))
        return {"kind": kind, "batch": batch, "nq": nq, "nkv": nkv, "d": d,
                "page": rng.choice([32, 64, 256]), "ctx_min": max(1, hi // 32), "ctx_max": hi}
    if kind == "gqa_prefill":
        nq, nkv, d = rng.choice(HEADS)
        batch = rng.choice([1, 1, 2])
        window = _log(rng, 2, 2011)
        most = min(16384, 2011 * 5000 * 32 * 128 // (nq * d * batch * window) + window // 2)
        return {"kind": kind, "batch": batch, "nq": nq, "nkv": nkv, "d": d,
                "page": rng.choice([32, 64, 256]), "seq": _log(rng, window, max(most, window)),
                "window": window}
    if kind == "mla_decode":
        batch = _log(rng, 1, 16)
        hi = _log(rng, 64, min(65536, 131072 // batch))
        return {"kind": kind, "batch": batch, "heads": rng.choice([128, 128, 64, 32]),
                "page": rng.choice([64, 256]), "ctx_min": max(1, hi // rng.choice([1, 8])),
                "ctx_max": hi}
    if kind == "mla_prefill":
        window = _log(rng, 2, 512)
        heads = rng.choice([128, 128, 64, 32])
        most = min(16384, 301 * 4247 * 128 // (heads * window) + window // 2)
        return {"kind": kind, "batch": 1, "heads": heads, "page": rng.choice([64, 256]),
                "seq": _log(rng, window, max(most, window)), "window": window}
    if kind == "dsa_decode":
        batch = rng.choice([1, 1, 2, 4])
        return {"kind": kind, "batch": batch, "heads": rng.choice([128, 64]),
                "page": rng.choice([64, 256]), "seq": _log(rng, 3000, 131072 // batch)}
    if kind == "position_free":
        nq, nkv, d = rng.choice(HEADS[:3])
        queries = rng.choice([1, 1, rng.randint(2, 4), _log(rng, 5, 250)])
        keys = _log(rng, max(64, queries), min(32768, 250 * 8003 // queries))
        return {"kind": kind, "nq": nq, "nkv": nkv, "d": d,
                "dtype": rng.choice(["bf16", "bf16", "f16", "f32"]), "keys": keys,
                "queries": queries}
    if kind == "spill_reload":
        page = rng.choice([64, 256])
        nkv, d = rng.choice([(8, 128), (4, 128), (3, 64)])
        layers = rng.randint(1, 4)
        pages = _log(rng, 4, 512 * 64 // (page * layers))
        return {"kind": kind, "layers": layers, "pages": pages, "page": page, "nkv": nkv, "d": d}
    if kind == "attend_spilled":
        nq, nkv, d = rng.choice(HEADS)
        page = rng.choice([64, 256])
        seq = _log(rng, 1100, 32801)
        return {"kind": kind, "nq": nq, "nkv": nkv, "d": d, "page": page, "seq": seq,
                "spilled": rng.randint(1, max(1, seq * 2 // (5 * page)))}
    if kind == "decoder_prefill":
        return {"kind": kind, "tokens": _log(rng, 6, 512)}
    return {"kind": kind, "prompt": _log(rng, 6, 900), "steps": rng.randint(4, 16)}


# ---- inputs -------------------------------------------------------------------


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(1000003 + seed)


def _randn(g: torch.Generator, *shape, std: float = 1.0, dtype=torch.bfloat16) -> torch.Tensor:
    """Normal values drawn in pieces (no fp32 copy of a large tensor)."""
    out = torch.empty(shape, dtype=dtype, device=DEV)
    flat = out.view(-1)
    step = 1 << 24
    for i in range(0, flat.numel(), step):
        n = min(step, flat.numel() - i)
        flat[i:i + n] = torch.randn(n, generator=g, device=DEV) * std
    return out


def _lengths(case: dict) -> list[int]:
    """Context lengths of a batch: the longest, the shortest, and the rest
    uniform between them.  Sizes belong to the case, so they do not depend on
    the seed."""
    lo, hi, n = case["ctx_min"], case["ctx_max"], case["batch"]
    r = random.Random(n * 1000003 + hi * 31 + lo)
    mid = [r.randint(lo, hi) for _ in range(n)]
    mid[0] = hi
    if n > 1:
        mid[-1] = lo
    return mid


def _paged(lengths: list[int], page: int, seed: int):
    """(slots, block table [B, max_pages] int32, lengths int32): pages at
    shuffled pool slots, as requests that come and go leave them."""
    per = [-(-n // page) for n in lengths]
    slots = sum(per)
    perm = torch.randperm(slots, generator=torch.Generator().manual_seed(seed)).tolist()
    table = torch.zeros((len(lengths), max(per)), dtype=torch.int32)
    at = 0
    for b, n in enumerate(per):
        table[b, :n] = torch.tensor(perm[at:at + n], dtype=torch.int32)
        at += n
    return slots, table.to(DEV), torch.tensor(lengths, dtype=torch.int32, device=DEV)


def _gqa_decode_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    page, nkv, d = case["page"], case["nkv"], case["d"]
    slots, table, ctx = _paged(_lengths(case), page, seed)
    vb = min(page, 32)
    return {"q": _randn(g, case["batch"], case["nq"], d, std=2.0),
            "k": _randn(g, slots, nkv, page, d),
            "v": _randn(g, slots, nkv, page // vb, d, vb), "table": table, "ctx": ctx}


def _gqa_cache_inputs(case: dict, seed: int, batch: int, window: int) -> dict:
    g = _gen(seed)
    seq, nkv, d = case["seq"], case["nkv"], case["d"]
    return {"k": _randn(g, batch, nkv, seq, d), "v": _randn(g, batch, nkv, seq, d),
            "q": _randn(g, batch, case["nq"], window, d, std=2.0)}


def _mla_inputs(case: dict, seed: int, batch: int, window: int) -> dict:
    g = _gen(seed)
    h = case["heads"]
    return {"q_nope": _randn(g, batch, h, window, DN), "q_rope": _randn(g, batch, h, window, ROPE),
            "w_uk": _randn(g, h, DN, LATENT, std=0.05), "w_uv": _randn(g, h, LATENT, DV, std=0.05)}


def _dsa_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    b, s, h = case["batch"], case["seq"], case["heads"]
    slots, table, ctx = _paged([s] * b, case["page"], seed)
    return {"keys": _randn(g, b, s, INDEX_DIM), "q_idx": _randn(g, b, INDEX_HEADS, INDEX_DIM),
            "w_head": torch.randn((b, INDEX_HEADS), generator=g, device=DEV) * INDEX_HEADS ** -0.5,
            "q_lat": _randn(g, b, h, LATENT + ROPE), "lat": _randn(g, slots, case["page"],
                                                                  LATENT + ROPE),
            "table": table, "ctx": ctx}


def _position_free_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    dt = DTYPES[case["dtype"]]
    n, tq, d = case["keys"], case["queries"], case["d"]
    pages = n + n // 4 + 8  # the pool also holds other requests' tokens
    ids = torch.randperm(pages, generator=torch.Generator().manual_seed(seed))[:n]
    half = d // 2
    inv = THETA ** (torch.arange(half, dtype=torch.float32, device=DEV) / half)
    ang = torch.arange(n, dtype=torch.float32, device=DEV)[:, None] / inv
    return {"q": _randn(g, 1, case["nq"], tq, d, std=2.0, dtype=dt),
            "k": _randn(g, pages, case["nkv"], 1, d, dtype=dt),
            "v": _randn(g, pages, case["nkv"], 1, d, dtype=dt),
            "table": ids.to(torch.int32).to(DEV),
            "kpos": torch.arange(n, dtype=torch.int32, device=DEV),
            "qpos": torch.arange(n - tq, n, dtype=torch.int32, device=DEV),
            "cos": torch.cos(ang), "sin": torch.sin(ang)}


def _weights(cfg: DecoderConfig, g: torch.Generator) -> dict[str, torch.Tensor]:
    """Random weights under the Hugging Face Llama names."""
    h, i, hd = cfg.hidden_size, cfg.intermediate_size, cfg.head_dim
    nq, nkv = cfg.num_attention_heads, cfg.num_key_value_heads
    ones = torch.ones(h, dtype=torch.bfloat16, device=DEV)
    w = {"model.embed_tokens.weight": _randn(g, cfg.vocab_size, h, std=0.02),
         "model.norm.weight": ones}
    for n in range(cfg.num_hidden_layers):
        p = f"model.layers.{n}"
        for name, rows, cols in (("self_attn.q_proj", nq * hd, h), ("self_attn.k_proj", nkv * hd, h),
                                 ("self_attn.v_proj", nkv * hd, h), ("self_attn.o_proj", h, nq * hd),
                                 ("mlp.gate_proj", i, h), ("mlp.up_proj", i, h),
                                 ("mlp.down_proj", h, i)):
            w[f"{p}.{name}.weight"] = _randn(g, rows, cols, std=0.02)
        w[f"{p}.input_layernorm.weight"] = w[f"{p}.post_attention_layernorm.weight"] = ones
    return w


def _decoder_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    cfg = DecoderConfig()
    n = case["tokens"] if case["kind"] == "decoder_prefill" else case["prompt"] + case["steps"]
    return {"cfg": cfg, "weights": _weights(cfg, g),
            "tokens": torch.randint(0, cfg.vocab_size, (1, n), generator=g, device=DEV)}


def _cache(layers: int, page: int) -> PagedKVCache:
    return PagedKVCache(layers, 1 << 62, page_positions=page, device=torch.device(DEV))


# ---- the interface ----------------------------------------------------------------


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "gqa_decode":
        st = _gqa_decode_inputs(case, seed)
    elif kind == "gqa_prefill":
        st = _gqa_cache_inputs(case, seed, case["batch"], case["window"])
        st["kv"] = _cache(1, case["page"])
        st["kv"].append(0, st.pop("k"), st.pop("v"))
    elif kind == "mla_decode":
        st = _mla_inputs(case, seed, case["batch"], 1)
        st["q_nope"], st["q_rope"] = st["q_nope"][:, :, 0], st["q_rope"][:, :, 0]
        slots, st["table"], st["ctx"] = _paged(_lengths(case), case["page"], seed)
        st["lat"] = _randn(_gen(seed + 77), slots, case["page"], LATENT + ROPE)
        st["w_uk"], st["w_uv"] = ops.pack_head_weights(st["w_uk"]), ops.pack_head_weights(st["w_uv"])
    elif kind == "mla_prefill":
        st = _mla_inputs(case, seed, case["batch"], case["window"])
        st["kv"] = _cache(1, case["page"])
        st["kv"].append_latent(0, _randn(_gen(seed + 77), case["batch"], case["seq"],
                                         LATENT + ROPE))
        st["w_uk"], st["w_uv"] = ops.pack_head_weights(st["w_uk"]), ops.pack_head_weights(st["w_uv"])
    elif kind == "dsa_decode":
        st = _dsa_inputs(case, seed)
    elif kind == "position_free":
        st = _position_free_inputs(case, seed)
    elif kind == "spill_reload":
        g = _gen(seed)
        st = {"kv": _cache(case["layers"], case["page"]),
              "pages": [(n, i) for n in range(case["layers"]) for i in range(case["pages"])]}
        shape = (1, case["nkv"], case["pages"] * case["page"], case["d"])
        for n in range(case["layers"]):
            st["kv"].append(n, _randn(g, *shape), _randn(g, *shape))
        st["kv"].arena.reserve(len(st["pages"]) * st["kv"].page_nbytes + (1 << 20))
    elif kind == "attend_spilled":
        st = _gqa_cache_inputs(case, seed, 1, 1)
        kv = st["kv"] = _cache(1, case["page"])
        kv.append(0, st.pop("k"), st.pop("v"))
        count = min(case["spilled"], case["seq"] // case["page"])
        kv.arena.reserve(count * kv.page_nbytes + (1 << 20))
        kv.spill([(0, i) for i in range(count)])
    else:
        st = _decoder_inputs(case, seed)
        st["model"] = PagedDecoder(st["cfg"], st.pop("weights"), device=torch.device(DEV))
        st["kv"] = st["model"].new_cache()
        if kind == "decoder_decode":
            n = st["start"] = case["prompt"]
            st["model"].forward(st["tokens"][:, :n], st["kv"], last_only=True)
            st["step_logits"] = torch.empty((1, st["cfg"].vocab_size), device=DEV)
            st["graph"], st["tok"], _ = st["model"].capture_decode(
                st["kv"], n + case["steps"], logits=st["step_logits"])
            st["out"] = torch.empty((case["steps"], st["cfg"].vocab_size), device=DEV)
    st["kind"] = kind
    return st


def run(st: dict):
    kind = st["kind"]
    if kind == "gqa_decode":
        return ops.paged_gqa_decode(st["q"], st["k"], st["v"], st["table"], st["ctx"])
    if kind == "gqa_prefill":
        return st["kv"].attend_prefill(0, st["q"])
    if kind == "mla_decode":
        return ops.mla_absorbed_decode(st["q_nope"], st["q_rope"], st["lat"], st["table"],
                                       st["ctx"], st["w_uk"], st["w_uv"],
                                       scale=(DN + ROPE) ** -0.5)
    if kind == "mla_prefill":
        return st["kv"].attend_mla_prefill(0, st["q_nope"], st["q_rope"], st["w_uk"], st["w_uv"],
                                           (DN + ROPE) ** -0.5)
    if kind == "dsa_decode":
        scores = ops.dsa_index_scores(st["q_idx"], st["w_head"], st["keys"], st["ctx"],
                                      scale=INDEX_DIM ** -0.5)
        sel, sel_lens = ops.dsa_topk(scores, st["ctx"], TOPK)
        out = ops.mla_sparse_decode(st["q_lat"], st["lat"], st["table"], sel, sel_lens,
                                    scale=(DN + ROPE) ** -0.5)
        return {"scores": scores, "sel": sel, "out": out}
    if kind == "position_free":
        return ops.position_free_paged_attention(
            st["q"], st["k"], st["v"], st["table"], st["kpos"], st["qpos"], st["cos"], st["sin"],
            scale=st["q"].shape[-1] ** -0.5)
    if kind == "spill_reload":
        kv = st["kv"]
        kv.spill(st["pages"])
        kv.reload(st["pages"])
        return [kv.gather(n) for n in range(kv.num_layers)]
    if kind == "attend_spilled":
        return st["kv"].attend(0, st["q"])
    if kind == "decoder_prefill":
        st["kv"].trim(0)
        return st["model"].forward(st["tokens"], st["kv"], last_only=True)
    kv, tokens, out = st["kv"], st["tokens"], st["out"]
    kv.trim(st["start"])
    for i in range(out.shape[0]):
        st["tok"].copy_(tokens[:, st["start"] + i:st["start"] + i + 1])
        st["graph"].replay()
        kv.advance(1)
        out[i].copy_(st["step_logits"][0])
    return out


def _decoder_work(tokens: int, before: int) -> dict:
    cfg = DecoderConfig()
    keys = sum(before + i + 1 for i in range(tokens))
    layer = cfg.param_count - cfg.vocab_size * cfg.hidden_size
    kv = cfg.num_key_value_heads * cfg.head_dim * 4 * cfg.num_hidden_layers
    return {"flops": 2.0 * layer * tokens
            + 4.0 * cfg.num_attention_heads * cfg.head_dim * keys * cfg.num_hidden_layers,
            "layer_bytes": 2.0 * layer, "kv_token": float(kv),
            "head_flops": 2.0 * cfg.vocab_size * cfg.hidden_size,
            "head_bytes": 2.0 * cfg.vocab_size * cfg.hidden_size + 4.0 * cfg.vocab_size}


def work(case: dict) -> dict:
    """Bytes and flops of one pass: every input once, every output once."""
    kind = case["kind"]
    if kind == "gqa_decode":
        n = sum(_lengths(case))
        qo = 4 * case["batch"] * case["nq"] * case["d"]
        return {"bytes": 4 * n * case["nkv"] * case["d"] + qo,
                "flops": 4 * n * case["nq"] * case["d"]}
    if kind in ("gqa_prefill", "mla_prefill"):
        b, s, w = case["batch"], case["seq"], case["window"]
        pairs = b * (w * s - w * (w - 1) // 2)
        if kind == "gqa_prefill":
            return {"bytes": 4 * b * (s * case["nkv"] + w * case["nq"]) * case["d"],
                    "flops": 4 * pairs * case["nq"] * case["d"]}
        h = case["heads"]
        weights = h * LATENT * (DN + DV)
        return {"bytes": 2 * (b * s * (LATENT + ROPE) + weights + b * w * h * (DN + ROPE + DV)),
                "flops": 2 * pairs * h * (2 * LATENT + ROPE) + 2 * b * w * weights}
    if kind == "mla_decode":
        b, h, n = case["batch"], case["heads"], sum(_lengths(case))
        weights = h * LATENT * (DN + DV)
        return {"bytes": 2 * (n * (LATENT + ROPE) + weights + b * h * (DN + ROPE + DV)),
                "flops": 2 * n * h * (2 * LATENT + ROPE) + 2 * b * weights}
    if kind == "dsa_decode":
        b, s, h = case["batch"], case["seq"], case["heads"]
        rows = min(s, TOPK)
        return {"bytes": b * (s * (2 * INDEX_DIM + 4) + 4 * TOPK
                              + 2 * (rows * (LATENT + ROPE) + h * (2 * LATENT + ROPE))),
                "flops": b * (2 * s * INDEX_HEADS * INDEX_DIM + 2 * rows * h * (2 * LATENT + ROPE))}
    if kind == "position_free":
        n, tq, nq, nkv, d = (case[k] for k in ("keys", "queries", "nq", "nkv", "d"))
        e = 4 if case["dtype"] == "f32" else 2
        pairs = tq * n - tq * (tq - 1) // 2
        return {"bytes": n * (2 * e * nkv * d + 8 + 4 * d) + 2 * e * nq * tq * d,
                "flops": 4 * pairs * nq * d}
    if kind == "spill_reload":
        # over the host link twice; on the device read, written, and gathered
        page = 4 * case["page"] * case["nkv"] * case["d"]
        return {"bytes": 6 * case["layers"] * case["pages"] * page, "flops": 0}
    if kind == "attend_spilled":
        return {"bytes": 4 * (case["seq"] * case["nkv"] + case["nq"]) * case["d"],
                "flops": 4 * case["seq"] * case["nq"] * case["d"]}
    if kind == "decoder_prefill":
        w = _decoder_work(case["tokens"], 0)
        return {"bytes": w["layer_bytes"] + w["head_bytes"] + 2 * w["kv_token"] * case["tokens"],
                "flops": w["flops"] + w["head_flops"]}
    n, p = case["steps"], case["prompt"]
    w = _decoder_work(n, p)
    keys = sum(p + i + 1 for i in range(n))
    return {"bytes": n * (w["layer_bytes"] + w["head_bytes"]) + w["kv_token"] * keys,
            "flops": w["flops"] + n * w["head_flops"]}


def tolerance(case: dict):
    """bf16 and fp16 results carry one rounding of their own (2^-9, 2^-12) and
    the softmax weights' rounding before them; about four times what separates
    the path from ``exact`` (see there)."""
    kind = case["kind"]
    if kind == "spill_reload":
        return "exact"
    if kind in ("decoder_prefill", "decoder_decode"):
        return {"rel": 0.03, "max": 0.2}  # bf16 roundings of 30 layers
    if kind == "position_free" and case["dtype"] == "f32":
        return {"rel": 1e-5, "max": 4e-4}
    if kind == "position_free" and case["dtype"] == "f16":
        return {"rel": 2e-3, "max": 2e-2}
    return {"rel": 1e-2, "max": 0.1}


# ---- 64-bit results ---------------------------------------------------------------


def _softmax_out(q, k, v, scale, first: int | None = None):
    """q [H, T, D], k [H or 1, S, D], v: softmax(q k^T scale) v in 64 bits; with
    ``first`` query t sees keys up to first + t."""
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) * scale
    if first is not None:
        at = torch.arange(s.shape[1], device=s.device)[:, None] + first
        s.masked_fill_(torch.arange(s.shape[2], device=s.device)[None, :] > at, -math.inf)
    return torch.matmul(torch.softmax(s, -1), v)


def _gqa64(q, k, v, scale, first=None):
    """q [NQ, T, D] over k, v [NKV, S, D], one kv head at a time."""
    nkv = k.shape[0]
    g = q.shape[0] // nkv
    return torch.cat([_softmax_out(q[j * g:(j + 1) * g].double(), k[j:j + 1].double(),
                                   v[j:j + 1].double(), scale, first) for j in range(nkv)])


def _exact_decoder(case: dict, seed: int) -> torch.Tensor:
    st = _decoder_inputs(case, seed)
    cfg, w, tokens = st["cfg"], st["weights"], st["tokens"][0]
    n, hd, nq, nkv = tokens.numel(), cfg.head_dim, cfg.num_attention_heads, cfg.num_key_value_heads
    half = hd // 2
    inv = 1.0 / cfg.rope_theta ** (torch.arange(half, device=DEV).double() / half)
    ang = torch.arange(n, device=DEV).double()[:, None] * inv
    cos, sin = ang.cos(), ang.sin()

    def norm(x):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + cfg.rms_norm_eps)

    def rope(x):
        a, b = x[..., :half], x[..., half:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    x = w["model.embed_tokens.weight"][tokens].double()
    for layer in range(cfg.num_hidden_layers):
        m = {k: w[f"model.layers.{layer}.{k}.weight"].double().t().contiguous() for k in
             ("self_attn.q_proj", "self_attn.k_proj", "self_attn.v_proj", "self_attn.o_proj",
              "mlp.gate_proj", "mlp.up_proj", "mlp.down_proj")}
        h = norm(x)
        q = rope((h @ m["self_attn.q_proj"]).view(n, nq, hd).transpose(0, 1))
        k = rope((h @ m["self_attn.k_proj"]).view(n, nkv, hd).transpose(0, 1))
        v = (h @ m["self_attn.v_proj"]).view(n, nkv, hd).transpose(0, 1)
        x = x + _gqa64(q, k, v, hd ** -0.5, 0).transpose(0, 1).reshape(n, -1) @ m["self_attn.o_proj"]
        h = norm(x)
        x = x + (torch.nn.functional.silu(h @ m["mlp.gate_proj"]) * (h @ m["mlp.up_proj"])) \
            @ m["mlp.down_proj"]
    if case["kind"] == "decoder_prefill":
        x = x[-1:]
    else:
        x = x[case["prompt"]:]
    out = norm(x) @ w["model.embed_tokens.weight"].double().t().contiguous()
    return out[None] if case["kind"] == "decoder_prefill" else out


def _exact_mla(q_nope, q_rope, w_uk, w_uv, lat, first):
    """[H, T, .] queries over latent rows [S, 576], one head at a time."""
    out = []
    keys, values = lat.double(), lat[:, :LATENT].double()
    for h in range(q_nope.shape[0]):
        q = torch.cat([q_nope[h].double() @ w_uk[h].double(), q_rope[h].double()], -1)
        c = _softmax_out(q[None], keys[None], values[None], (DN + ROPE) ** -0.5, first)[0]
        out.append(c @ w_uv[h].double())
    return torch.stack(out)


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "gqa_decode":
        st = _gqa_decode_inputs(case, seed)
        out = []
        for b, n in enumerate(_lengths(case)):
            ids = st["table"][b, :-(-n // case["page"])].long()
            k = st["k"][ids].permute(1, 0, 2, 3).reshape(case["nkv"], -1, case["d"])[:, :n]
            v = st["v"][ids].permute(1, 0, 2, 4, 3).reshape(case["nkv"], -1, case["d"])[:, :n]
            out.append(_gqa64(st["q"][b][:, None], k, v, case["d"] ** -0.5)[:, 0])
        return torch.stack(out)
    if kind in ("gqa_prefill", "attend_spilled"):
        batch, window = (case["batch"], case["window"]) if kind == "gqa_prefill" else (1, 1)
        st = _gqa_cache_inputs(case, seed, batch, window)
        return torch.stack([_gqa64(st["q"][b], st["k"][b], st["v"][b], case["d"] ** -0.5,
                                   case["seq"] - window) for b in range(batch)])
    if kind == "mla_decode":
        st = _mla_inputs(case, seed, case["batch"], 1)
        slots, table, _ = _paged(_lengths(case), case["page"], seed)
        lat = _randn(_gen(seed + 77), slots, case["page"], LATENT + ROPE)
        out = []
        for b, n in enumerate(_lengths(case)):
            rows = lat[table[b, :-(-n // case["page"])].long()].reshape(-1, LATENT + ROPE)[:n]
            out.append(_exact_mla(st["q_nope"][b], st["q_rope"][b], st["w_uk"], st["w_uv"], rows,
                                  None)[:, 0])
        return torch.stack(out)
    if kind == "mla_prefill":
        st = _mla_inputs(case, seed, case["batch"], case["window"])
        lat = _randn(_gen(seed + 77), case["batch"], case["seq"], LATENT + ROPE)
        return torch.stack([_exact_mla(st["q_nope"][b], st["q_rope"][b], st["w_uk"], st["w_uv"],
                                       lat[b], case["seq"] - case["window"])
                            for b in range(case["batch"])])
    if kind == "dsa_decode":
        st = _dsa_inputs(case, seed)
        scores, outs = [], []
        for b in range(case["batch"]):
            s = torch.relu(st["keys"][b].double() @ st["q_idx"][b].double().t().contiguous())
            s = (s * INDEX_DIM ** -0.5) @ st["w_head"][b].double()
            sel = torch.topk(s, min(TOPK, s.numel())).indices.sort().values
            rows = st["lat"][st["table"][b].long()].reshape(-1, LATENT + ROPE)[sel].double()
            scores.append(s)
            outs.append(_softmax_out(st["q_lat"][b].double()[None], rows[None],
                                     rows[None, :, :LATENT], (DN + ROPE) ** -0.5)[0])
        # ties and last-place differences of the scores may order keys otherwise
        return {"scores": torch.stack(scores), "sel": None, "out": torch.stack(outs)}
    if kind == "position_free":
        st = _position_free_inputs(case, seed)
        ids, half = st["table"].long(), case["d"] // 2
        k = st["k"][ids, :, 0].transpose(0, 1)
        v = st["v"][ids, :, 0].transpose(0, 1)
        a, b = k[..., :half].double(), k[..., half:].double()
        cos, sin = st["cos"].double(), st["sin"].double()
        # a rotated key is a value of the element type
        k = torch.cat([a * cos - b * sin, b * cos + a * sin], -1).to(st["q"].dtype)
        return _gqa64(st["q"][0], k, v, case["d"] ** -0.5, case["keys"] - case["queries"])[None]
    if kind == "spill_reload":
        return None
    return _exact_decoder(case, seed)
