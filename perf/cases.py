"""The work a user of this framework has it do, as cases that can be timed and
checked: decode and prefill attention over the paged KV pool, decoder layers
of the Qwen3 shapes at decode and prefill sizes, a whole decode step, and the
sampler, each through the package's public modules.  Decode work runs as the
model runner runs it, recorded once per batch size by HipGraphRunner and
replayed; prefill work runs eagerly.

Kinds (the "kind" of a case):
  attn_decode   Attention: KV store of one token per sequence + paged decode
  attn_prefix   the same where some sequences share their first pages
  attn_prefill  Attention: KV store + causal attention of whole prompts
  attn_chunk    Attention: prompt chunks over pages already in the pool
  decode        Qwen3 decoder layers, one token per sequence, to the final norm
  prefill       a Qwen3 decoder layer over one step's prompts, to the final norm
  step          the whole decode step of a model, to its logits
  sample        Sampler over a batch's logits
"""
import math
import random
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path("xixi-vllm_amd").resolve()))

from xvllm.config import QWEN3_0_6B, QWEN3_8B, QWEN3_32B, Qwen3Shape  # noqa: E402
from xvllm.cuda_graph import HipGraphRunner  # noqa: E402
from xvllm.kv_pool import KVPool  # noqa: E402
from xvllm.layers.attention import (Attention, AttnInputs, AttnMetadata, CascadePlan,  # noqa: E402
                                    attention_context)
from xvllm.models import Qwen3ForCausalLM  # noqa: E402
from xvllm.prefix_cache import cascade_groups  # noqa: E402
from xvllm.sampler import Sampler, reserve_workspace  # noqa: E402

D = 128  # head_dim of every supported shape
SHAPES = {"0.6B": QWEN3_0_6B, "8B": QWEN3_8B, "32B": QWEN3_32B}
HEADS = {"0.6B": (16, 8), "8B": (32, 8), "32B": (64, 8)}  # query heads, kv heads
KV_SCALE = 0.025  # fp8 pages: |x| <= 448 * 0.025 = 11.2 is representable
BF16, F64 = torch.bfloat16, torch.float64


def listed():
    return [
        # one user chatting: the smallest call there is, launch latency and the split over the chip
        dict(name="attn_decode_one", kind="attn_decode", model="8B", rows=1, lo=1937, hi=1937, kv="bf16", block=16, mix=1),
        # the headline decode batch: 64 sequences of uneven context
        dict(name="attn_decode_64", kind="attn_decode", model="8B", rows=64, lo=512, hi=4096, kv="bf16", block=16, mix=2),
        # the same on the fp8 page format, with the larger model's eight query heads per kv head
        dict(name="attn_decode_fp8", kind="attn_decode", model="32B", rows=48, lo=700, hi=6000, kv="fp8", block=16, mix=3),
        # long contexts, half of the sequences with one system prompt in shared pages
        dict(name="attn_shared_prefix", kind="attn_prefix", model="32B", rows=32, shared=4096, members=16, lo=4200, hi=12000,
             block=16, mix=4),
        # a prefill step of new prompts
        dict(name="attn_prefill_prompts", kind="attn_prefill", model="8B", rows=16, lo=128, hi=2048, mix=5),
        # chunked prefill: 512-token chunks over what the pool already holds of each prompt
        dict(name="attn_prefill_chunks", kind="attn_chunk", model="8B", rows=16, q=512, lo=0, hi=1536, kv="bf16", block=16, mix=6),
        # decoder layers of a decode step with packed decode weights, the headline batch ...
        dict(name="layers_decode_64", kind="decode", model="8B", layers=2, rows=64, lo=512, hi=2048, packed=True, mix=7),
        # ... and a full serving batch, where the weights are used by more rows
        dict(name="layers_decode_200", kind="decode", model="8B", layers=2, rows=200, lo=128, hi=1536, packed=True, mix=8),
        # a decoder layer over one 8192-token prefill budget, one prompt
        dict(name="layer_prefill_8192", kind="prefill", model="8B", rows=1, lo=8192, hi=8192, mix=9),
        # a small model's whole decode step for a handful of users: hundreds of short kernels
        dict(name="step_small_model", kind="step", model="0.6B", rows=8, lo=128, hi=512, packed=True, mix=10),
        # sampling of a serving batch: temperature 0.7, top-k 50, top-p 0.9 over peaked logits
        dict(name="sample_top_k", kind="sample", rows=256, mode="top_k", spread=2.5),
        # nucleus sampling without top-k over flat logits
        dict(name="sample_top_p", kind="sample", rows=32, mode="top_p", spread=1.43),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attn_decode", "attn_decode", "attn_prefix", "attn_prefill", "attn_chunk", "decode", "decode",
                       "prefill", "step", "sample"])
    mix = rng.randrange(1 << 20)
    model = rng.choice(["0.6B", "8B", "32B"])
    if kind == "attn_decode":
        rows = _log_int(rng, 1, 256)
        hi = min(_log_int(rng, 64, 16384), 262144 // rows)
        return dict(kind=kind, model=model, rows=rows, lo=max(1, hi // 8), hi=hi, kv=rng.choice(["bf16", "fp8"]),
                    block=rng.choice([16, 16, 256]), mix=mix)
    if kind == "attn_prefix":
        rows = rng.randint(4, 40)
        shared = 16 * rng.randint(32, 384)
        return dict(kind=kind, model=model, rows=rows, shared=shared, members=rng.randint(2, min(rows, 16)),
                    lo=shared + 1, hi=shared + rng.randint(64, 4096), block=16, mix=mix)
    if kind == "attn_prefill":
        rows = _log_int(rng, 1, 48)
        hi = min(_log_int(rng, 48, 8192), 16384 // rows)
        return dict(kind=kind, model=rng.choice(["0.6B", "8B"]), rows=rows, lo=max(1, hi // 8), hi=hi, mix=mix)
    if kind == "attn_chunk":
        rows = _log_int(rng, 1, 24)
        q = min(_log_int(rng, 8, 4096), 8192 // rows)
        hi = min(_log_int(rng, 64, 12288), 49152 // rows)
        return dict(kind=kind, model=rng.choice(["0.6B", "8B"]), rows=rows, q=q, lo=hi // 4, hi=hi,
                    kv=rng.choice(["bf16", "fp8"]), block=rng.choice([16, 16, 256]), mix=mix)
    if kind == "decode":
        return dict(kind=kind, model=model, layers=2, rows=_log_int(rng, 1, 256), lo=64, hi=_log_int(rng, 128, 1536),
                    packed=rng.random() < 0.7, mix=mix)
    if kind == "prefill":
        rows = _log_int(rng, 1, 16)
        hi = min(_log_int(rng, 24, 4096), 8192 // rows)
        return dict(kind=kind, model=rng.choice(["0.6B", "8B"]), rows=rows, lo=max(1, hi // 4), hi=hi, mix=mix)
    if kind == "step":
        return dict(kind=kind, model="0.6B", rows=_log_int(rng, 1, 64), lo=32, hi=_log_int(rng, 64, 1024),
                    packed=rng.random() < 0.7, mix=mix)
    return dict(kind="sample", rows=_log_int(rng, 1, 400), mode=rng.choice(["greedy", "top_k", "top_p", "top_k_any", "min_p"]),
                spread=round(rng.uniform(1.0, 4.0), 2))


# ---------------------------------------------------------------- sizes of a case
def _lens(c):
    """Tokens of each sequence (attn_chunk: tokens already in the pool)."""
    r = random.Random(c["mix"])
    return [r.randint(c["lo"], c["hi"]) for _ in range(c["rows"])]


def _cfg(c):
    """The model of a "decode", "prefill" or "step" case: the layers asked
    for; layer cases stop at the final norm, so their vocabulary is small."""
    s = SHAPES[c["model"]]
    whole = c["kind"] == "step"
    return Qwen3Shape(s.hidden_size, s.num_attention_heads, s.num_key_value_heads, s.head_dim, s.intermediate_size,
                      s.num_hidden_layers if whole else c.get("layers", 1), vocab_size=s.vocab_size if whole else 8192,
                      max_position_embeddings=16384)


def _pairs(q, k):
    """Visible (query, key) pairs of a causal chunk of q queries ending a run of k keys."""
    return q * (k - q) + q * (q + 1) // 2


def work(c):
    if c["kind"] == "sample":
        return {"bytes": c["rows"] * (151936 * 2 + 28), "flops": 0}
    lens = _lens(c)
    n = len(lens)
    if c["kind"].startswith("attn"):
        hq, hkv = HEADS[c["model"]]
        kvb = 1 if c.get("kv") == "fp8" else 2
        tok = 2 * hkv * D  # K and V elements of a token
        if c["kind"] in ("attn_decode", "attn_prefix"):
            keys = sum(lens)
            read = keys - (c["members"] - 1) * c["shared"] if c["kind"] == "attn_prefix" else keys
            return {"bytes": read * tok * kvb + n * (2 * hq * D + tok) * 2, "flops": 4 * hq * D * keys}
        if c["kind"] == "attn_prefill":
            return {"bytes": sum(lens) * (2 * hq * D * 2 + tok * 4), "flops": 4 * hq * D * sum(_pairs(s, s) for s in lens)}
        q = c["q"]
        return {"bytes": sum(s + q for s in lens) * tok * kvb + n * q * (2 * hq * D + tok) * 2,
                "flops": 4 * hq * D * sum(_pairs(q, s + q) for s in lens)}
    s = _cfg(c)
    h, hq, hkv, inter, layers = (s.hidden_size, s.num_attention_heads, s.num_key_value_heads, s.intermediate_size,
                                 s.num_hidden_layers)
    weights = layers * (h * (hq + 2 * hkv) * D + hq * D * h + 3 * h * inter)
    head = s.vocab_size * h if c["kind"] == "step" else 0
    tok = 2 * hkv * D
    if c["kind"] == "prefill":
        t = sum(lens)
        return {"bytes": weights * 2 + t * (2 * h + tok * layers) * 2,
                "flops": 2 * t * weights + 4 * hq * D * layers * sum(_pairs(k, k) for k in lens)}
    return {"bytes": (weights + head) * 2 + layers * sum(lens) * tok * 2 + n * (2 * h + (head and s.vocab_size)) * 2,
            "flops": 2 * n * (weights + head) + 4 * hq * D * layers * sum(lens)}


def tolerance(c):
    """Whole numbers (token ids) are exact.  bf16 results: an attention output
    measures 2.0e-3 to 2.9e-3 (2-norm) off the 64-bit value, two layers 6.4e-3,
    a whole model, whose roundings travel through 28 layers, 1.6e-2; another
    order of the sums is off by as much again, in another direction."""
    if c["kind"] == "sample":
        return "exact"
    if c["kind"].startswith("attn"):
        return {"rel": 1e-2, "max": 0.1}
    return {"rel": 3e-2 if c["kind"] == "step" else 2e-2, "max": 0.3}


# ---------------------------------------------------------------- inputs, from the seed alone
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, std=1.0):
    return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std).to(BF16)


def _tables(c, lens, seed):
    """Block tables of sequences of `lens` tokens: a random permutation of a
    pool a quarter larger than needed (members of a shared prefix start with
    the same blocks); rows past a sequence's end hold -1."""
    bs = c.get("block", 16)
    need = [-(-s // bs) for s in lens]
    pool = max(4, int(1.25 * sum(need)) + 1)
    perm = np.random.RandomState(seed % (1 << 31)).permutation(pool).astype(np.int32)
    bt = np.full((len(lens), max(need)), -1, np.int32)
    at = 0
    for b, k in enumerate(need):
        first = c["shared"] // bs if c["kind"] == "attn_prefix" and 0 < b < c["members"] else 0
        bt[b, :first] = bt[0, :first]
        bt[b, first:k] = perm[at : at + k - first]
        at += k - first
    return bt, pool, bs


def _slots(bt, bs, spans):
    return np.concatenate([bt[b, np.arange(i, j) // bs] * bs + np.arange(i, j) % bs for b, (i, j) in enumerate(spans)])


def _dev(a, dt=torch.int32):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dt)


def _inputs(c, seed):
    """Everything a pass reads, as plain tensors."""
    g = _gen(seed)
    if c["kind"] == "sample":
        v = 151936
        return dict(logits=_randn(g, c["rows"], v, std=c["spread"]),
                    u=torch.rand(c["rows"], generator=g, device="cuda", dtype=torch.float32))
    lens = _lens(c)
    n = len(lens)
    chunk = c["kind"] == "attn_chunk"
    prefill = c["kind"] in ("attn_prefill", "attn_chunk", "prefill")
    total = [s + c["q"] for s in lens] if chunk else lens
    bt, blocks, bs = _tables(c, total, seed)
    spans = [(s, t) for s, t in zip(lens, total)] if chunk else [(0, t) if prefill else (t - 1, t) for t in total]
    x = dict(total=total, spans=spans, bt=bt, blocks=blocks, block=bs, slots=_dev(_slots(bt, bs, spans)),
             pos=_dev(np.concatenate([np.arange(i, j) for i, j in spans]), torch.int64))
    rows = sum(j - i for i, j in spans)
    if c["kind"].startswith("attn"):
        hq, hkv = HEADS[c["model"]]
        # q, k and v as views of one fused projection output, as the decoder has them
        qkv = _randn(g, rows, (hq + 2 * hkv) * D)
        x.update(q=qkv[:, : hq * D], k=qkv[:, hq * D : (hq + hkv) * D].view(rows, hkv, D),
                 v=qkv[:, (hq + hkv) * D :].view(rows, hkv, D), hq=hq, hkv=hkv, layers=1)
    else:
        s = _cfg(c)
        x.update(ids=torch.randint(0, s.vocab_size, (rows,), generator=g, device="cuda"), cfg=s, hq=s.num_attention_heads,
                 hkv=s.num_key_value_heads, layers=s.num_hidden_layers)
    x["pool"] = None
    if c["kind"] not in ("attn_prefill", "prefill"):
        x["pool"] = torch.randn((2, x["layers"], blocks, x["hkv"], bs, D), generator=g, device="cuda", dtype=BF16)
    return x


def _weights(c, seed):
    """name -> tensor of a Qwen3 shape's weights, N(0, 0.02), norm weights 1 + N(0, 0.1)."""
    s = _cfg(c)
    g = _gen(seed + 7919)
    h, i = s.hidden_size, s.intermediate_size
    q, kv = s.num_attention_heads * D, s.num_key_value_heads * D
    w = {"model.embed_tokens": _randn(g, s.vocab_size, h, std=1.0), "lm_head": _randn(g, s.vocab_size, h, std=0.02),
         "model.norm.weight": 1 + _randn(g, h, std=0.1)}
    for k in range(s.num_hidden_layers):
        p = f"model.layers.{k}."
        w[p + "self_attn.qkv_proj"] = _randn(g, q + 2 * kv, h, std=0.02)
        w[p + "self_attn.o_proj"] = _randn(g, h, q, std=0.02)
        w[p + "mlp.gate_up_proj"] = _randn(g, 2 * i, h, std=0.02)
        w[p + "mlp.down_proj"] = _randn(g, h, i, std=0.02)
        for name, size in (("input_layernorm", h), ("post_attention_layernorm", h), ("self_attn.q_norm", D),
                           ("self_attn.k_norm", D)):
            w[p + name + ".weight"] = 1 + _randn(g, size, std=0.1)
    return w


# ---------------------------------------------------------------- what a user's program has in hand
def _recorded(rows, body):
    """`body` recorded for this batch size, as the model runner records its decode step."""
    with torch.inference_mode():
        graphs = HipGraphRunner([rows], torch.device("cuda"))
        graphs.capture(body)
    return graphs


def _prepare_sample(c, seed):
    x = _inputs(c, seed)
    rows, v = x["logits"].shape
    full = lambda value, dt: torch.full((rows,), value, dtype=dt, device="cuda")  # noqa: E731
    mode = c["mode"]
    reserve_workspace(x["logits"].device, rows, v)
    temps = full(0.0 if mode == "greedy" else 1.0 if mode == "top_p" else 0.7, torch.float32)
    args = dict(all_greedy=mode == "greedy", uniforms=x["u"])
    if mode in ("top_k", "top_k_any"):
        args.update(top_ks=full(50, torch.int32), top_ps=full(0.9, torch.float32), use_top_k=True, use_top_p=True,
                    max_top_k=50 if mode == "top_k" else 0)
    elif mode == "top_p":
        args.update(top_ps=full(0.95, torch.float32), use_top_p=True)
    elif mode == "min_p":
        args.update(min_ps=full(0.05, torch.float32), use_min_p=True)
    sampler = Sampler()
    return dict(rows=rows, keep=(x, temps, args), graphs=_recorded(rows, lambda _: sampler(x["logits"], temps, **args)))


def prepare(c, seed):
    if c["kind"] == "sample":
        return _prepare_sample(c, seed)
    x = _inputs(c, seed)
    fp8 = c.get("kv") == "fp8"
    cfg = x.get("cfg") or Qwen3Shape(x["hq"] * D, x["hq"], x["hkv"], D, 128, 1)
    pool = KVPool(cfg, num_blocks=x["blocks"], block_size=x["block"], device=torch.device("cuda"),
                  dtype=torch.float8_e4m3fn if fp8 else BF16, num_layers=x["layers"],
                  **(dict(k_scale=KV_SCALE, v_scale=KV_SCALE) if fp8 else {}))
    if x["pool"] is None:
        pool.kv_cache.zero_()
    else:
        pool.kv_cache.copy_((x["pool"] / KV_SCALE if fp8 else x["pool"]).transpose(3, 4))
        x["pool"] = None
    meta = AttnMetadata(kv_cache=pool.kv_cache, k_scale=pool.k_scale, v_scale=pool.v_scale)
    total, spans, bt = x["total"], x["spans"], _dev(x["bt"])
    if c["kind"] in ("attn_prefill", "attn_chunk", "prefill"):
        cu = lambda v: _dev(np.concatenate([[0], np.cumsum(v)]))  # noqa: E731
        q_lens = [j - i for i, j in spans]
        attn = AttnInputs(slot_mapping=x["slots"], is_prefill=True, cu_seqlens_q=cu(q_lens), cu_seqlens_k=cu(total),
                          max_seqlen_q=max(q_lens), max_seqlen_k=max(total),
                          block_tables=bt if c["kind"] == "attn_chunk" else None)
    else:
        plan = None
        if c["kind"] == "attn_prefix":
            pre, info, group_rows = cascade_groups(x["bt"], np.asarray(total), x["block"],
                                                   max_rows=128 // (x["hq"] // x["hkv"]), min_blocks=16, max_groups=4,
                                                   max_prefix_blocks=x["bt"].shape[1])
            plan = CascadePlan(_dev(pre), _dev(info), _dev(group_rows), 4, x["bt"].shape[1])
        attn = AttnInputs(slot_mapping=x["slots"], is_prefill=False, block_tables=bt, cache_seqlens=_dev(total),
                          cascade=plan)
    state = dict(meta=meta, attn=attn, pool=pool.kv_cache.view(torch.uint8) if fp8 else pool.kv_cache, rows=len(total))
    if c["kind"].startswith("attn"):
        layer = Attention(x["hq"], D, x["hkv"])
        state["body"] = lambda _: layer(x["q"], x["k"], x["v"], attn)
    else:
        was = torch.get_default_dtype()
        torch.set_default_dtype(BF16)
        try:
            with torch.device("cuda"):
                model = Qwen3ForCausalLM(cfg)
        finally:
            torch.set_default_dtype(was)
        with torch.no_grad():
            for name, p in _weights(c, seed).items():
                model.get_parameter(name).copy_(p)
        if c.get("packed"):
            model.pack_decode_weights()
        state["model"] = model
        if c["kind"] == "step":
            state["body"] = lambda _: model.compute_logits(model(x["ids"], x["pos"], attn))
        else:
            state["body"] = lambda _: model(x["ids"], x["pos"], attn)
    if not attn.is_prefill:
        with attention_context(meta):
            state["graphs"] = _recorded(len(total), state["body"])
    return state


def run(state):
    if "graphs" in state:
        out = state["graphs"].replay(state["rows"])[0]
    else:
        with torch.inference_mode(), attention_context(state["meta"]):
            out = state["body"](None)
    return out if "pool" not in state else (out, state["pool"])


# ---------------------------------------------------------------- the same in 64 bits, in plain torch
def _attend(q, k, v, shift):
    """q [Lq, Hq, D], k / v [Lk, Hkv, D]: query i sees keys j <= shift + i."""
    lq, hq, lk = q.shape[0], q.shape[1], k.shape[0]
    grp = hq // k.shape[1]
    out = torch.empty_like(q)
    hidden = None
    if lq > 1:
        hidden = torch.arange(lk, device=q.device)[None] > shift + torch.arange(lq, device=q.device)[:, None]
    for h in range(hq):
        s = q[:, h] @ k[:, h // grp].T / math.sqrt(D)
        if hidden is not None:
            s.masked_fill_(hidden, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, h // grp]
    return out


def _attention(x, q, k, v, cached):
    """All sequences' attention: each attends to its tokens already in the
    pool (cached(b, end) gives their k and v) and to this pass's own."""
    out, at = torch.empty_like(q), 0
    for b, (i, j) in enumerate(x["spans"]):
        kb, vb = k[at : at + j - i], v[at : at + j - i]
        if i:
            kc, vc = cached(b, i)
            kb, vb = torch.cat([kc, kb]), torch.cat([vc, vb])
        out[at : at + j - i] = _attend(q[at : at + j - i], kb, vb, i)
        at += j - i
    return out


def _cached(x, layer):
    def rows(b, end):
        bs = x["block"]
        ids = torch.from_numpy(x["bt"][b, : -(-end // bs)].astype(np.int64)).cuda()
        kv = x["pool"][:, layer, ids].to(F64).transpose(2, 3).reshape(2, -1, x["hkv"], D)[:, :end]
        return kv[0], kv[1]
    return rows


def _norm(x, w, eps=1e-6):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _rope(x, pos, theta):
    inv = theta ** (-torch.arange(0, D, 2, device=x.device, dtype=F64) / D)
    a = pos.to(F64)[:, None, None] * inv
    lo, hi = x[..., : D // 2], x[..., D // 2 :]
    return torch.cat([lo * a.cos() - hi * a.sin(), hi * a.cos() + lo * a.sin()], -1)


def exact(c, seed):
    if c["kind"] == "sample":
        return None
    x = _inputs(c, seed)
    if c.get("kv") == "fp8":  # what the pages hold, and what storing this pass's tokens leaves in them
        e4m3 = lambda t: (t / KV_SCALE).to(BF16).to(torch.float8_e4m3fn).to(F64) * KV_SCALE  # noqa: E731
        new = lambda t: (t.float() * (1 / KV_SCALE)).to(torch.float8_e4m3fn).to(F64) * KV_SCALE  # noqa: E731
        x["pool"] = e4m3(x["pool"])
    else:
        new = lambda t: t.to(F64)  # noqa: E731
    if c["kind"].startswith("attn"):
        rows = x["q"].shape[0]
        out = _attention(x, x["q"].to(F64).view(rows, x["hq"], D), new(x["k"]), new(x["v"]), _cached(x, 0))
        return out.reshape(rows, -1), None
    s, w = x["cfg"], _weights(c, seed)
    hq, hkv = x["hq"], x["hkv"]
    rows = x["ids"].shape[0]
    res = w["model.embed_tokens"][x["ids"]].to(F64)
    for k in range(s.num_hidden_layers):
        get = lambda name: w[f"model.layers.{k}.{name}"].to(F64)  # noqa: B023, E731
        qkv = _norm(res, get("input_layernorm.weight")) @ get("self_attn.qkv_proj").T
        q = _rope(_norm(qkv[:, : hq * D].view(rows, hq, D), get("self_attn.q_norm.weight")), x["pos"], s.rope_theta)
        kk = _rope(_norm(qkv[:, hq * D : (hq + hkv) * D].reshape(rows, hkv, D), get("self_attn.k_norm.weight")),
                   x["pos"], s.rope_theta)
        o = _attention(x, q, kk, qkv[:, (hq + hkv) * D :].view(rows, hkv, D), _cached(x, k))
        res = res + o.reshape(rows, -1) @ get("self_attn.o_proj").T
        gu = _norm(res, get("post_attention_layernorm.weight")) @ get("mlp.gate_up_proj").T
        gate, up = gu[:, : s.intermediate_size], gu[:, s.intermediate_size :]
        res = res + (torch.nn.functional.silu(gate) * up) @ get("mlp.down_proj").T
    hidden = _norm(res, w["model.norm.weight"].to(F64))
    return (hidden @ w["lm_head"].to(F64).T if c["kind"] == "step" else hidden), None
