"""Dense GEMMs of the decoder: up to 256 rows the gfx950 kernel that streams
the [N, K] weight in place (xv_stream_gemm: gate_up fused with SiLU-and-mul,
down and o as split-K partials for the norm that follows them, reference
src/compute/models/qwen3.py:64,115 feeding the norms of :150,:152, a decode
batch's qkv as partials for its norm + RoPE + KV store), above that
and for shapes it does not take PyTorch (hipBLASLt) with a split-K form for
down and o.  A model that was not packed streams down and o only where that
form splits (split_factor > 1), since its callers see PartialSums only there:
Qwen3-0.6B's two, Qwen3-8B's down up to 16 rows and its o at 17 to 48, and
Qwen3-32B's o up to 32 rows and at 65 to 80 stay on hipBLASLt.  A prefill
batch's qkv does at every size (attention reads its q, k and v as bf16).
pack_weight / dense_gemm are the older streamed form over packed
weight tiles (at most 64 rows), kept where the in-place kernel does not take
a shape: Qwen3-32B's gate_up (51200 x 5120) at 17 to 64 rows, 87 us at 32
rows against hipBLASLt's 98.

us of the products alone with the weights streamed from HBM, hipBLASLt -> in
place (gate_up with its SiLU; MI355X, graph replay, over 1 GB of weights cycled):
    Qwen3-8B    gate_up  M 8: 46.5 -> 31.0   M 64: 47.8 -> 34.6   M 200: 64.5 -> 54.9
                down     M 8: 22.1 -> 18.1   M 64: 23.6 -> 20.1   M 200: 34.6 -> 31.7
                o        M 8: 10.3 -> 8.0    M 64: 14.8 -> 9.6    M 200: 18.1 -> 16.6
                qkv      M 8: 15.7 -> 11.3   M 64: 18.0 -> 11.9   M 200: 26.8 -> 21.1 (4 partial sums)
    Qwen3-0.6B  gate_up  M 8: 10.3 -> 5.1    down M 8: 12.1 -> 4.0   o M 8: 9.7 -> 3.4

us that a decode layer takes longer with one of its products, and its
consumer, on hipBLASLt instead (recorded model bodies of 4 to 24 packed layers,
contexts of 64 tokens; runs of one side differ by up to 1 us, 3 at Qwen3-32B):
    Qwen3-0.6B  (58 .. 81 a layer)    qkv 3 .. 6   gate_up 2 .. 5    o -0.2 .. 2.7   down -2.2 .. 0
    Qwen3-8B    (118 .. 185)          qkv 5 .. 21  gate_up 7 .. 13   o -0.8 .. 2.7   down 1.4 .. 5.7
    Qwen3-32B   (235 .. 372)          qkv 10 .. 30 (no gate_up)      o 3 .. 13       down -0.4 .. 22
    hidden 2048, MLP 6144 (72 .. 106) qkv 0.5 .. 11  gate_up 1.5 .. 7  o 0.8 .. 3.8  down 0.5 .. 6.5
    hidden 2560, MLP 9728 (99 .. 156) (qkv not timed, no gate_up)      o 2 .. 11     down 4 .. 15
at M 72 to 256.  Only Qwen3-0.6B's down loses (packed models, above 72 rows:
from 96 rows on its 8 partial sums, written and read, are more bytes than the
weight), by less than its gate_up gains.  Up to 16 rows a gate_up that has a packed copy runs
in place too: Qwen3-32B 4 rows 2.9 us faster, 12 rows even, 16 rows 2.5 slower.

The split-K measurements below are the hipBLASLt path.

At decode batch sizes an [M, K] x [K, 4096] GEMM has few output tiles for 256
CUs: hipBLASLt runs Qwen3-8B's o_proj (K 4096) and down_proj (K 12288) at
1.4-2.7 TB/s between M 32 and 256.  Cut along K into P slices, the same
weights run as a batched GEMM with P times the tiles (one bmm over strided
views, no copies), each slice's fp32 product kept apart; the norm kernel
that consumes them sums the P partials, rounds to bf16 (the value the
unsplit GEMM would have written) and continues as fused_add_rmsnorm.  The
partials cost P x M x N x 4 bytes of extra reads in the norm, which the
table below charges against the GEMM's gain.

The split per shape and batch size is SPLIT_TABLE, measured for the Qwen3-8B
and Qwen3-32B weights; the first measurements, which set split_rule for other
shapes (MI355X, graph replay, more than 1 GB of weights cycled so that none is
served from the 256 MB last-level cache; us, unsplit -> split):

    down_proj  M 32: 28.2 -> 22.6 (P 4)   M 64: 37.5 -> 25.0 (P 4)
               M 128: 66.2 -> 27.3 (P 8)  M 256: 54.4 -> 36.0 (P 8)
               M 1, 8: no gain
    o_proj     M 1, 8: 15.3 -> 10.1 (P 4)  M 128: 24.2 -> 15.6 (P 8)
               M 32, 64, 256: gains below the partials' extra reads

On hipBLASLt gate_up stays unsplit (same measurement, bmm over the same views):
gate_up (K 4096, N 24576) M 32-128: 45-51 unsplit, no split faster; M 256:
65.5 -> 59.6 (P 2), less than its 50 MB of fp32 partials cost to write and
read back.
"""
from __future__ import annotations

import bisect
from typing import NamedTuple

import torch
import torch.nn.functional as F
from torch._subclasses.fake_tensor import FakeTensor


class PartialSums(NamedTuple):
    """fp32 partial products [P, M, N] of one split-K GEMM; their sum is the
    GEMM's output."""

    parts: torch.Tensor

    def materialize(self) -> torch.Tensor:
        """The bf16 [M, N] output of the unsplit GEMM (for callers outside
        the decoder's norm chain)."""
        return self.parts.sum(0).to(torch.bfloat16)


# The fastest K split per decode graph bucket (SPLIT_BUCKETS) for the o_proj
# and down_proj weights of Qwen3-8B ([4096, 4096], [4096, 12288]) and
# Qwen3-32B ([5120, 8192], [5120, 25600]), measured on MI355X by
# `python -m xvllm.layers.split_tune` (the GEMM plus the norm that sums its
# partials, graph replay, weights cycled past the last-level cache).
# hipBLASLt's kernel choice makes the best split jump between neighbouring
# sizes, so the table is taken as measured.  At Qwen3-32B's M 32 it runs
# o_proj unsplit (27.6 us against 54.2 at P 4) and down_proj at P 2 (80.1
# against 89.1 us).  Other shapes use split_rule.
SPLIT_BUCKETS = (1, 2, 4, 8, 16, 32, 48, 64, 80, 96, 112, 128, 144, 160, 176, 192, 208, 224, 240, 256)
SPLIT_TABLE = {
    (4096, 4096): (4, 4, 4, 4, 4, 1, 1, 2, 2, 2, 2, 2, 2, 4, 2, 4, 2, 4, 2, 4),
    (4096, 12288): (1, 1, 1, 1, 1, 4, 4, 4, 4, 4, 8, 8, 8, 8, 8, 8, 8, 8, 8, 8),
    (5120, 8192): (1, 1, 1, 1, 1, 1, 8, 8, 1, 2, 4, 2, 2, 8, 2, 8, 4, 8, 4, 8),
    (5120, 25600): (2, 2, 2, 2, 2, 2, 8, 8, 8, 4, 8, 8, 8, 8, 8, 8, 4, 8, 8, 8),
}


def split_rule(m: int, n: int, k: int) -> int:
    """K slices for a shape outside SPLIT_TABLE (the Qwen3-8B measurements
    above, generalised by K)."""
    if n > 8192 or k % (8 * 64):
        return 1
    if k >= 8192:
        return 4 if 32 <= m < 96 else 8 if 96 <= m <= 256 else 1
    if k >= 4096:
        return 4 if m <= 16 else 8 if 96 <= m <= 192 else 1
    return 1


def split_factor(m: int, n: int, k: int) -> int:
    """K slices for an [m, k] x [k, n] GEMM feeding a norm (1: no split):
    SPLIT_TABLE's entry for the smallest bucket of at least m rows, else
    split_rule; above 256 rows, 1."""
    if m < 1 or m > SPLIT_BUCKETS[-1]:
        return 1
    row = SPLIT_TABLE.get((n, k))
    if row is None:
        return split_rule(m, n, k)
    return row[bisect.bisect_left(SPLIT_BUCKETS, m)]


def linear_into_norm(x: torch.Tensor, w: torch.Tensor, split: bool = True):
    """x [M, K] @ w[N, K]^T for a consumer that accepts PartialSums (the
    residual add + RMSNorm of the next norm): the split-K partials when
    split_factor picks a split, else the plain bf16 product."""
    m, k = x.shape
    n = w.shape[0]
    p = split_factor(m, n, k) if split else 1
    if p == 1 or x.stride(1) != 1 or w.stride(1) != 1:
        return F.linear(x, w)
    xs, ws = split_k_views(x, w, p)
    return PartialSums(torch.bmm(xs, ws, out_dtype=torch.float32))


def split_k_views(x: torch.Tensor, w: torch.Tensor, p: int) -> tuple[torch.Tensor, torch.Tensor]:
    """Slice p of x [M, K] and of w [N, K] along K as batched-GEMM operands,
    views only: x -> [P, M, K/P], w -> [P, K/P, N] (w^T's slices)."""
    m, k = x.shape
    n = w.shape[0]
    return x.view(m, p, k // p).transpose(0, 1), w.view(n, p, k // p).permute(1, 2, 0)


# Output forms of xv_dense_gemm (csrc/dense_gemm.hip).
GEMM_BF16, GEMM_PARTS, GEMM_SILU_MUL = 0, 1, 2


class PackedWeight(NamedTuple):
    """A [N, K] weight in the tile order the decode GEMM kernel streams:
    16-row x 64-column tiles of 2 KB, each in the kernel's lane order (see
    pack_weight), row blocks outermost."""

    data: torch.Tensor  # bf16, N * K elements
    n: int
    k: int


def pack_weight(w: torch.Tensor) -> PackedWeight:
    """Pack w [N, K] (N % 16 == 0, K % 64 == 0) for dense_gemm: tile (nb, sg)
    holds, for lane l = 16 g + r (r < 16, g < 4), w[16 nb + r, 64 sg + 8 g + e]
    at 8 l + e and w[16 nb + r, 64 sg + 32 + 8 g + e] at 512 + 8 l + e."""
    n, k = w.shape
    if n % 16 or k % 64:
        raise ValueError(f"pack_weight: [{n}, {k}] is not a whole number of 16 x 64 tiles")
    t = w.reshape(n // 16, 16, k // 64, 2, 4, 8)  # [nb, r, sg, half, g, e]
    return PackedWeight(t.permute(0, 2, 3, 4, 1, 5).contiguous().view(-1), n, k)


def dense_gemm(x: torch.Tensor, w: PackedWeight, mode: int = GEMM_BF16, *, col_tiles: int = 4, waves: int = 4,
               parts: int = 1):
    """x [M, K] @ w^T on the weight-streaming gfx950 kernel (M <= 64), w packed
    by pack_weight.

    mode GEMM_BF16: bf16 [M, N].  GEMM_PARTS: PartialSums of a K split over
    `parts` ([P, M, N] fp32).  GEMM_SILU_MUL: w is the gate/up weight [2I, K]
    (gate rows first) and the result is bf16 silu(x w_gate^T) * (x w_up^T),
    [M, I], the two products rounded to bf16 first as the unfused GEMM stores
    them.  col_tiles x 16 weight rows per wave (1, 2 or 4; even for
    GEMM_SILU_MUL), `waves` (4 or 8) waves per workgroup over the same K.
    Raises on shapes or layouts the kernel does not take."""
    from .. import _C
    from .._torch_glue import ptr, require_bf16, require_cuda, stream_of

    require_cuda(x)
    require_bf16(x)
    require_bf16(w.data)
    m, k = x.shape
    n = w.n
    if x.stride(1) != 1:
        raise ValueError("dense_gemm: x needs unit stride along K")
    if w.k != k:
        raise ValueError(f"dense_gemm: x {tuple(x.shape)} and w [{w.n}, {w.k}] disagree on K")
    if w.data.numel() != w.n * w.k or not w.data.is_contiguous() or w.n % 16 or w.k % 64:
        raise ValueError(f"dense_gemm: packed weight holds {w.data.numel()} elements "
                         f"(contiguous: {w.data.is_contiguous()}), not whole 16 x 64 tiles of [{w.n}, {w.k}]")
    if mode == GEMM_PARTS:
        out = torch.empty((parts, m, n), dtype=torch.float32, device=x.device)
        os_, ps = n, m * n
    else:
        out = torch.empty((m, n // 2 if mode == GEMM_SILU_MUL else n), dtype=torch.bfloat16, device=x.device)
        os_, ps = out.shape[1], 0
    _C.check(
        _C.lib().xv_dense_gemm(ptr(x), x.stride(0), ptr(w.data), ptr(out), os_, ps, m, n, k, mode, col_tiles, waves,
                               parts, stream_of(x)),
        "xv_dense_gemm",
    )
    return PartialSums(out) if mode == GEMM_PARTS else out


def stream_parts(k: int) -> int:
    """K slices of a split-K product over a packed weight (the most of 8, 4,
    2, 1 that cut K into whole 4-step rounds)."""
    for p in (8, 4, 2, 1):
        if k % (p * 256) == 0:
            return p
    return 0


# Rows up to which a weight is streamed in place (xv_stream_gemm), and from a packed copy (xv_dense_gemm).
IN_PLACE_MAX_ROWS = 256
STREAM_MAX_ROWS = 64


def streamable(w: torch.Tensor, mode: int) -> bool:
    """Whether w [N, K] fits the shapes of the packed decode GEMMs:
    gate/up + SiLU with 2 tiles x 4 waves (2I % 128), split-K partials with
    1 tile x 8 waves (N % 128)."""
    n, k = w.shape
    if mode == GEMM_SILU_MUL:
        return n % 128 == 0 and k % 256 == 0
    return n % 128 == 0 and stream_parts(k) > 0


def stream_rows(x: torch.Tensor) -> bool:
    """Whether activations x [M, K] can take a packed decode GEMM: at most
    STREAM_MAX_ROWS rows, unit stride along K, 16-byte aligned rows."""
    return (0 < x.shape[0] <= STREAM_MAX_ROWS and x.stride(1) == 1 and x.stride(0) % 8 == 0
            and x.data_ptr() % 16 == 0)


def in_place_parts(m: int, n: int, k: int, mode: int) -> int:
    """Partial sums of an [m, k] x [k, n] product on the kernel that streams
    the [N, K] weight in place (xv_stream_gemm): 1 .. 8, or 0 where it does
    not take the shape (more than 256 rows, or a column count that does not
    divide evenly over the CUs)."""
    from .. import _C

    return _C.lib().xv_stream_gemm_parts(m, n, k, mode)


@torch.library.custom_op("xv::stream_gemm", mutates_args=())
def _stream_gemm(x: torch.Tensor, w: torch.Tensor, mode: int, parts: int) -> torch.Tensor:
    """x [M, K] against w [N, K] in place: fp32 [parts, M, N] partial sums
    (GEMM_PARTS) or bf16 silu(x w_gate^T) * (x w_up^T) [M, N / 2] (GEMM_SILU_MUL)."""
    from .. import _C
    from .._torch_glue import aligned16, ptr, require_bf16, require_cuda, stream_of

    require_cuda(x, w)
    require_bf16(x, w)
    m, k = x.shape
    n = w.shape[0]
    if w.shape[1] != k:
        raise ValueError(f"stream_gemm: x {tuple(x.shape)} and w {tuple(w.shape)} disagree on K")
    if x.stride(1) != 1 or x.stride(0) % 8 or x.stride(0) < k or not aligned16(x):  # (expanded and overlapping rows: stride < K)
        x = x.clone(memory_format=torch.contiguous_format)
    if w.stride(1) != 1:
        raise ValueError("stream_gemm: w needs unit stride along K")
    if mode == GEMM_PARTS:
        out = torch.empty((parts, m, n), dtype=torch.float32, device=x.device)
        os_, ps = n, m * n
    else:
        out = torch.empty((m, n // 2), dtype=torch.bfloat16, device=x.device)
        os_, ps = n // 2, 0
    _C.check(
        _C.lib().xv_stream_gemm(ptr(x), x.stride(0), ptr(w), w.stride(0), ptr(out), os_, ps, m, n, k, mode, parts,
                                stream_of(x)),
        "xv_stream_gemm",
    )
    return out


@_stream_gemm.register_fake
def _stream_gemm_fake(x, w, mode, parts):
    m, n = x.shape[0], w.shape[0]
    if mode == GEMM_PARTS:
        return x.new_empty((parts, m, n), dtype=torch.float32)
    return x.new_empty((m, n // 2))


def _streams_in_place(w: torch.Tensor) -> bool:
    """Whether w [N, K] has the layout xv_stream_gemm reads: rows of unit
    stride, whole (not expanded, not overlapping) and 16-byte aligned."""
    if w.stride(1) != 1 or w.stride(0) % 8 or w.stride(0) < w.shape[1] or w.storage_offset() % 8:
        return False
    # a storage need not start aligned (memory imported from elsewhere); a traced tensor has no address
    return isinstance(w, FakeTensor) or w.data_ptr() % 16 == 0


def stream_operand(x: torch.Tensor, w: torch.Tensor, packed, mode: int, *, internal: bool = False):
    """What streamed_silu_mul / streamed_into_norm read the weight w [N, K]
    from for activations x: w itself where the in-place kernel takes the
    shape, else its packed copy (if it has one) up to STREAM_MAX_ROWS rows,
    else None (the library GEMM; also under torch.compile).  `packed` is the operand a packed model
    holds, None for a model that was not packed.  Such a model's callers get
    PartialSums only where linear_into_norm splits, so its products into a
    norm stream only there (unless they stay `internal` to the layer); and with gradients asked of x or w the library
    keeps the product (streaming has no backward; a packed model's batches of
    up to STREAM_MAX_ROWS rows are inference only)."""
    if torch.compiler.is_compiling():  # the shape rule is a C call, which a compiler's trace cannot hold
        return None
    if x.dim() != 2 or not 0 < x.shape[0] <= IN_PLACE_MAX_ROWS:  # first: a prefill step's layers ask three times each
        return None
    if not x.is_cuda or x.device != w.device or x.dtype != torch.bfloat16 or w.dtype != torch.bfloat16:
        return None
    m, k = x.shape
    n = w.shape[0]
    if packed is None and mode == GEMM_PARTS and not internal and split_factor(m, n, k) == 1:
        return None
    if (packed is None or m > STREAM_MAX_ROWS) and torch.is_grad_enabled() and (x.requires_grad or w.requires_grad):
        return None
    if _streams_in_place(w) and in_place_parts(m, n, k, mode) > 0:
        return w
    return packed if isinstance(packed, PackedWeight) and stream_rows(x) else None


def streamed_silu_mul(x: torch.Tensor, w) -> torch.Tensor:
    """silu(x w_gate^T) * (x w_up^T) of a short batch, bf16 [M, I]; w is the
    [2I, K] weight or its PackedWeight."""
    if isinstance(w, PackedWeight):
        return dense_gemm(x, w, GEMM_SILU_MUL, col_tiles=2, waves=4)
    return torch.ops.xv.stream_gemm(x, w, GEMM_SILU_MUL, 1)


def streamed_into_norm(x: torch.Tensor, w) -> PartialSums:
    """x @ w^T of a short batch as split-K PartialSums for the next residual
    add + RMSNorm; w is the [N, K] weight or its PackedWeight.  A packed
    weight's K is cut P = 8 ways where it allows; up to 32 rows, K slices
    under 1024 elements are halved instead (measured: Qwen3-8B o_proj at
    M 8, P 4 7.3 us against P 8 7.8; down_proj P 8 at every M)."""
    if isinstance(w, PackedWeight):
        p = stream_parts(w.k)
        if x.shape[0] <= 32 and w.k // p < 1024 and p > 1:
            p //= 2
        return dense_gemm(x, w, GEMM_PARTS, col_tiles=1, waves=8, parts=p)
    p = in_place_parts(x.shape[0], w.shape[0], x.shape[1], GEMM_PARTS)
    return PartialSums(torch.ops.xv.stream_gemm(x, w, GEMM_PARTS, p))
