"""Shared seeded input builders for the parity tests."""
from __future__ import annotations

import numpy as np
import torch


def gen(seed: int) -> torch.Generator:
    return torch.Generator().manual_seed(seed)


def randn_bf16(shape, g, std=1.0, mean=0.0):
    """fp32 draw then bf16 cast (how every synthetic input here is made)."""
    return (torch.randn(shape, generator=g) * std + mean).to(torch.bfloat16)


def f32(t: torch.Tensor) -> np.ndarray:
    return t.detach().to("cpu", torch.float32).numpy()


def make_paged(ctx_lens, num_blocks_pool, hkv, d, g, page=16, fill_nan=True):
    """Random-permutation block tables over a pool; unused pool rows hold NaN
    so any read past a sequence end shows up in the output."""
    ctx_lens = [int(c) for c in ctx_lens]
    need = [(c + page - 1) // page for c in ctx_lens]
    assert sum(need) <= num_blocks_pool
    perm = torch.randperm(num_blocks_pool, generator=g).tolist()
    max_blocks = max(max(need), 1)
    bt = torch.full((len(ctx_lens), max_blocks), -1, dtype=torch.int32)
    o = 0
    for b, n in enumerate(need):
        bt[b, :n] = torch.tensor(perm[o : o + n], dtype=torch.int32)
        o += n
    kc = randn_bf16((num_blocks_pool, page, hkv, d), g)
    vc = randn_bf16((num_blocks_pool, page, hkv, d), g)
    if fill_nan:
        valid = torch.zeros(num_blocks_pool, page, dtype=torch.bool)
        for b, c in enumerate(ctx_lens):
            for p in range(c):
                valid[bt[b, p // page], p % page] = True
        kc[~valid] = float("nan")
        vc[~valid] = float("nan")
    return kc, vc, bt, torch.tensor(ctx_lens, dtype=torch.int32)


# ---- the kernels of the in-place streaming GEMM (xv_stream_gemm)
STREAM_CLASSES = (16, 32, 64, 128, 256)  # the most rows of each row class


def stream_kernel(lib, m, n, k, mode):
    """(mode, row class, 16-row tiles per workgroup) of the kernel that takes
    an m x n x k product, None where it is not taken: the fewest tiles that
    keep the call within 256 workgroups, gate/up up to 16 rows two."""
    parts = lib.xv_stream_gemm_parts(m, n, k, mode)
    if parts == 0:
        return None
    tiles = n // 16
    sizes = (1, 2, 4, 5, 6, 8, 10) if mode == 1 else (2,) if m <= 16 else (2, 4, 6, 8)
    bnt = next(b for b in sizes if tiles % b == 0 and (tiles // b * parts <= 256 or (mode == 2 and m <= 16)))
    return mode, next(c for c in STREAM_CLASSES if m <= c), bnt


def stream_kernel_shapes(lib):
    """kernel -> (n, k), for every kernel a shape reaches: slices of an odd
    number of stages (128 elements up to 64 rows, else 64), at least 21, twice
    the deepest ring and one."""
    shapes = {}
    for mode in (1, 2):
        for m in STREAM_CLASSES:
            for parts in (8, 4, 2, 1) if mode == 1 else (1,):
                for stages in (21, 45, 93):
                    k = stages * (128 if m <= 64 else 64) * parts
                    for bnt in (1, 2, 4, 5, 6, 8, 10):
                        for blocks in (256, 240, 232, 224):
                            n = blocks // parts * bnt * 16
                            if blocks % parts == 0 and lib.xv_stream_gemm_parts(m, n, k, mode) == parts:
                                shapes.setdefault(stream_kernel(lib, m, n, k, mode), (n, k))
    return shapes
