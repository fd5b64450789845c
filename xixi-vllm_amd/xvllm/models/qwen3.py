"""Qwen3 dense decoder wired onto the xvllm operator API, one GPU (the
reference's tp=1, pp=1 case of src/compute/models/qwen3.py:44-238).

Per layer: input RMSNorm (fused with the residual add after layer 0), fused
qkv GEMM, per-head q/k RMSNorm + NeoX RoPE (one kernel, `xv::qk_norm_rope`),
`vllm::attention` (KV store + paged decode / prefill), o GEMM, fused add +
RMSNorm, gate_up GEMM, SiLU-and-mul, down GEMM.  Batches of up to 256 rows
stream gate_up (with the SiLU-and-mul) in place (xv_stream_gemm), decode
batches also qkv, as partials into the norm + RoPE + KV store kernel, and
down and o as split-K partials into the next norm: a packed model at every
size, others where the library's product would split too.  Larger batches and
the products and shapes outside this run on PyTorch (hipBLASLt).  Weights are plain
tensors (random init for the benchmarks; the reference's checkpoint loader is
out of scope).
"""
from __future__ import annotations

import torch
import torch.nn.functional as F
from torch import nn

from ..config import head_dim as _head_dim
from ..config import rope_theta as _rope_theta
from ..layers import Attention, AttnInputs, RMSNorm, RotaryEmbedding
from ..layers.attention import kv_cache_of, kv_scales
from ..layers.linear import (GEMM_PARTS, GEMM_SILU_MUL, STREAM_MAX_ROWS, in_place_parts, linear_into_norm, pack_weight,
                             stream_operand, stream_rows, streamable, streamed_into_norm, streamed_silu_mul)
from ..layers import ops as _ops  # noqa: F401  (registers the custom ops)
from ..sampler import sample


class StalePackedWeights(RuntimeError):
    """A weight was written or replaced after pack_decode_weights copied it:
    the streamed decode GEMMs would read the old values."""


def _weight_stamp(*params) -> tuple:
    return tuple((p._version, p.data_ptr()) for p in params)


def _check_stamp(module, stamp: tuple, *params) -> None:
    """Raise when a packed weight's source changed since it was packed
    (in-place writes through the Parameter bump its version; assigning a new
    tensor moves its data pointer).  Writes through `.data` bypass the version
    counter and are not seen."""
    if _weight_stamp(*params) != stamp:
        raise StalePackedWeights(f"{type(module).__name__}: weights changed after pack_decode_weights; "
                                 "call model.pack_decode_weights(False) then pack_decode_weights() again "
                                 "(outside graph capture; re-capture the decode graphs)")


def _needs_copy(w: torch.Tensor, mode: int) -> bool:
    """Whether decode batches of up to STREAM_MAX_ROWS rows stream w from a
    packed copy: the in-place kernel does not take the shape at every size
    (its rule has one case up to 16 rows and one above)."""
    return any(in_place_parts(m, *w.shape, mode) == 0 for m in (16, STREAM_MAX_ROWS))


def _packed_copy(p: nn.Parameter, mode: int):
    """The packed copy of a weight, None where the in-place kernel streams the weight itself."""
    return pack_weight(p.data) if _needs_copy(p, mode) else None


def _is_observed(attn: nn.Module) -> bool:
    """Whether something besides Attention.forward sees the arguments of a
    call of `attn`: hooks, or a module or a forward put in its place."""
    return bool(type(attn) is not Attention or "forward" in vars(attn) or attn._forward_hooks or attn._forward_pre_hooks
                or nn.modules.module._global_forward_hooks or nn.modules.module._global_forward_pre_hooks)


class Qwen3MLP(nn.Module):
    def __init__(self, hidden: int, inter: int):
        super().__init__()
        self.gate_up_proj = nn.Parameter(torch.empty(2 * inter, hidden))  # [gate; up] (linear.py:297-304)
        self.down_proj = nn.Parameter(torch.empty(hidden, inter))
        self.split_k = True
        self._copies = None  # pack(): the packed copies of (gate_up, down), None for one read in place

    def forward(self, x):
        """SiLU-MLP; the down GEMM may return PartialSums (split-K) for the
        next residual add + RMSNorm."""
        if not self.split_k:
            return F.linear(torch.ops.vllm.silu_and_mul(F.linear(x, self.gate_up_proj)), self.down_proj)
        if self._copies is not None and stream_rows(x):
            _check_stamp(self, self._stamp, self.gate_up_proj, self.down_proj)
        gate_up, down = self.packed or (None, None)
        w = stream_operand(x, self.gate_up_proj, gate_up, GEMM_SILU_MUL)
        if w is not None:
            act = streamed_silu_mul(x, w)
        else:
            act = torch.ops.vllm.silu_and_mul(F.linear(x, self.gate_up_proj))
        w = stream_operand(act, self.down_proj, down, GEMM_PARTS)
        return streamed_into_norm(act, w) if w is not None else linear_into_norm(act, self.down_proj)

    @property
    def packed(self):
        """The (gate_up, down) decode operands of pack(), None before it."""
        if self._copies is None:
            return None
        return self._copies[0] or self.gate_up_proj, self._copies[1] or self.down_proj

    def pack(self, enabled: bool = True):
        if not enabled:
            self._copies = None
        elif self._copies is None and streamable(self.gate_up_proj, GEMM_SILU_MUL) and streamable(self.down_proj,
                                                                                                    GEMM_PARTS):
            self._copies = (_packed_copy(self.gate_up_proj, GEMM_SILU_MUL), _packed_copy(self.down_proj, GEMM_PARTS))
            self._stamp = _weight_stamp(self.gate_up_proj, self.down_proj)


class Qwen3Attention(nn.Module):
    def __init__(self, cfg, layer_id: int):
        super().__init__()
        self.num_heads = cfg.num_attention_heads
        self.num_kv_heads = cfg.num_key_value_heads
        self.head_dim = _head_dim(cfg)
        self.q_size = self.num_heads * self.head_dim
        self.kv_size = self.num_kv_heads * self.head_dim
        self.qkv_proj = nn.Parameter(torch.empty(self.q_size + 2 * self.kv_size, cfg.hidden_size))
        self.o_proj = nn.Parameter(torch.empty(cfg.hidden_size, self.q_size))
        self.q_norm = RMSNorm(self.head_dim, cfg.rms_norm_eps)
        self.k_norm = RMSNorm(self.head_dim, cfg.rms_norm_eps)
        self.rotary_emb = RotaryEmbedding(self.head_dim, self.head_dim, cfg.max_position_embeddings, _rope_theta(cfg))
        self.attn = Attention(self.num_heads, self.head_dim, self.num_kv_heads, layer_id=layer_id)
        self.eps = cfg.rms_norm_eps
        self.split_k = True
        self._copies = None  # pack(): the packed copy of (o_proj,), None if read in place

    def forward(self, positions, hidden, attn: AttnInputs):
        """qkv -> q/k norm + RoPE -> attention -> o GEMM (PartialSums when
        split along K, for post_attention_layernorm)."""
        w = None if attn.is_prefill or not self.split_k else stream_operand(hidden, self.qkv_proj, None, GEMM_PARTS,
                                                                            internal=True)
        if w is not None:
            # decode: the qkv partial sums go into norm + RoPE + KV store
            qkv = streamed_into_norm(hidden, w)
            q = self._norm_rope_store_parts(positions, qkv.parts, attn.slot_mapping)
            q = k = v = q.view(q.shape[0], self.q_size)
            if _is_observed(self.attn):
                _, k, v = self._views(qkv.materialize())
            # Attention itself takes k and v from the cache (no slots to store at) and reads neither argument
            o = self.attn(q, k, v, attn._replace(slot_mapping=None))
        elif not attn.is_prefill:
            # decode: norm + RoPE + KV store in one kernel, attention reads the cache
            q, k, v = self._split_norm_rope_store(positions, F.linear(hidden, self.qkv_proj), attn.slot_mapping)
            o = self.attn(q.view(q.shape[0], self.q_size), k, v, attn._replace(slot_mapping=None))
        else:
            q, k, v = self._split_norm_rope(positions, F.linear(hidden, self.qkv_proj))
            o = self.attn(q.view(q.shape[0], self.q_size), k, v, attn)
        if not self.split_k:
            return F.linear(o, self.o_proj)
        if self._copies is not None and stream_rows(o):
            _check_stamp(self, self._stamp, self.o_proj)
        w = stream_operand(o, self.o_proj, self.packed_o, GEMM_PARTS)
        return streamed_into_norm(o, w) if w is not None else linear_into_norm(o, self.o_proj)

    @property
    def packed_o(self):
        """The o_proj decode operand of pack(), None before it."""
        return None if self._copies is None else self._copies[0] or self.o_proj

    def pack(self, enabled: bool = True):
        if not enabled:
            self._copies = None
        elif self._copies is None and streamable(self.o_proj, GEMM_PARTS):
            self._copies = (_packed_copy(self.o_proj, GEMM_PARTS),)
            self._stamp = _weight_stamp(self.o_proj)

    def _views(self, qkv):
        t = qkv.shape[0]
        q = qkv[:, : self.q_size].view(t, self.num_heads, self.head_dim)
        k = qkv[:, self.q_size : self.q_size + self.kv_size].view(t, self.num_kv_heads, self.head_dim)
        v = qkv[:, self.q_size + self.kv_size :].view(t, self.num_kv_heads, self.head_dim)
        return q, k, v

    def _split_norm_rope_store(self, positions, qkv, slot_mapping):
        q, k, v = self._views(qkv)
        k_cache, v_cache = kv_cache_of(self.attn.layer_id)
        ks, vs = kv_scales()
        q = torch.ops.xv.qk_norm_rope_store(
            q, k, v, self.q_norm.weight, self.k_norm.weight, self.eps, positions, self.rotary_emb.cos_sin_cache,
            k_cache, v_cache, slot_mapping, ks, vs,
        )
        return q, k, v

    def _norm_rope_store_parts(self, positions, parts, slot_mapping):
        k_cache, v_cache = kv_cache_of(self.attn.layer_id)
        ks, vs = kv_scales()
        t = parts.shape[1]  # positions and slots may come from buffers of a larger batch
        return torch.ops.xv.qk_norm_rope_store_parts(
            parts, self.num_heads, self.q_norm.weight, self.k_norm.weight, self.eps, positions.reshape(-1)[:t],
            self.rotary_emb.cos_sin_cache, k_cache, v_cache, slot_mapping.reshape(-1)[:t], ks, vs,
        )

    def _split_norm_rope(self, positions, qkv):
        """split -> per-head q/k RMSNorm -> RoPE (reference qwen3.py:117-128),
        the two norms and the rotation as one kernel reading the qkv views."""
        q, k, v = self._views(qkv)
        q, k = torch.ops.xv.qk_norm_rope(
            q, k, self.q_norm.weight, self.k_norm.weight, self.eps, positions, self.rotary_emb.cos_sin_cache
        )
        return q, k, v


class Qwen3DecoderLayer(nn.Module):
    def __init__(self, cfg, layer_id: int):
        super().__init__()
        self.self_attn = Qwen3Attention(cfg, layer_id)
        self.mlp = Qwen3MLP(cfg.hidden_size, cfg.intermediate_size)
        self.input_layernorm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps)
        self.post_attention_layernorm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps)

    def forward(self, positions, hidden, residual, attn: AttnInputs):
        """(hidden, residual) -> (hidden, residual) as the reference layer
        (qwen3.py:149-153), except that the returned hidden may be the
        PartialSums of the split-K down GEMM: the next layer's input norm (or
        the final norm) consumes them; PartialSums.materialize() gives the
        bf16 tensor."""
        hidden, residual = self.input_layernorm(hidden, residual)
        hidden = self.self_attn(positions, hidden, attn)
        hidden, residual = self.post_attention_layernorm(hidden, residual)
        return self.mlp(hidden), residual


class Qwen3Model(nn.Module):
    def __init__(self, cfg):
        super().__init__()
        self.embed_tokens = nn.Parameter(torch.empty(cfg.vocab_size, cfg.hidden_size))
        self.layers = nn.ModuleList([Qwen3DecoderLayer(cfg, i) for i in range(cfg.num_hidden_layers)])
        self.norm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps)

    def forward(self, input_ids, positions, attn: AttnInputs):
        h, residual = F.embedding(input_ids, self.embed_tokens), None
        for layer in self.layers:
            h, residual = layer(positions, h, residual, attn)
        return self.norm(h, residual)[0]


class Qwen3ForCausalLM(nn.Module):
    def __init__(self, cfg):
        super().__init__()
        self.config = cfg
        self.model = Qwen3Model(cfg)
        self.lm_head = nn.Parameter(torch.empty(cfg.vocab_size, cfg.hidden_size))

    def forward(self, input_ids, positions, attn: AttnInputs):
        return self.model(input_ids, positions, attn)

    def set_split_k(self, enabled: bool):
        """Split-K for o_proj / down_proj at decode batch sizes (on by default)."""
        for m in self.modules():
            if isinstance(m, (Qwen3Attention, Qwen3MLP)):
                m.split_k = enabled
        return self

    @torch.no_grad()
    def pack_decode_weights(self, enabled: bool = True):
        """Fix every layer's gate_up, down and o weights for the streamed
        decode GEMMs.  Weights whose shape the in-place kernel takes at every
        decode size are read where they are; the others (the Qwen3-32B
        shape's gate_up: 524 MB per layer) get a packed copy for batches of
        up to STREAM_MAX_ROWS rows, packed_decode_bytes() in all.  Layers that have
        copies keep them (the graphs captured over them stay valid).
        enabled=False drops them: only when no captured graph still uses
        them.  Call once the weights are final: the copies do not follow later
        writes (an eager forward raises StalePackedWeights when a fixed
        weight was written in place or replaced since).  Size the KV pool
        after packing, or pass packed_decode_bytes() as
        KVPool.auto_num_blocks' reserve_bytes."""
        for m in self.modules():
            if isinstance(m, (Qwen3Attention, Qwen3MLP)):
                m.pack(enabled)
        return self

    def packed_decode_bytes(self) -> int:
        """Bytes pack_decode_weights adds (the weights it copies)."""
        total = 0
        for m in self.modules():
            if isinstance(m, Qwen3MLP) and streamable(m.gate_up_proj, GEMM_SILU_MUL) and streamable(m.down_proj,
                                                                                                  GEMM_PARTS):
                pairs = ((m.gate_up_proj, GEMM_SILU_MUL), (m.down_proj, GEMM_PARTS))
            elif isinstance(m, Qwen3Attention) and streamable(m.o_proj, GEMM_PARTS):
                pairs = ((m.o_proj, GEMM_PARTS),)
            else:
                continue
            total += sum(w.numel() * w.element_size() for w, mode in pairs if _needs_copy(w, mode))
        return total

    def compute_logits(self, hidden):
        return F.linear(hidden, self.lm_head)

    def argmax(self, hidden):
        """Greedy ids (reference vocab_parallel.py:180-216): argmax of the bf16
        logits, lowest id on ties, by the sampler kernel."""
        logits = self.compute_logits(hidden)
        return sample(logits, None, all_greedy=True)

    @torch.no_grad()
    def random_init_(self, std: float = 0.02, seed: int = 0):
        """Weights ~ N(0, std) (norm weights 1), drawn on the parameters' device."""
        g = torch.Generator(device=self.lm_head.device).manual_seed(seed)
        for name, p in self.named_parameters():
            if name.endswith("norm.weight"):
                p.fill_(1.0)
            else:
                p.normal_(0.0, std, generator=g)
        return self
