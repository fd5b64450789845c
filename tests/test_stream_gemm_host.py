"""The rule of the in-place streaming GEMM (xv_stream_gemm_parts) and its
argument checks, on the CPU: every shape it takes cuts into whole tiles,
stages and 192 (gate/up) or 224 to 256 workgroups, the calls around its edges are refused
before anything is launched, every kernel the rule picks exists, and CPU inputs and long batches keep the library path."""
import random

import pytest
import torch
from helpers import STREAM_CLASSES, stream_kernel, stream_kernel_shapes

INVALID, A = 1, 1 << 20  # hipErrorInvalidValue; an aligned address no call reaches


@pytest.fixture(scope="module")
def lib():
    from xvllm import _C

    return _C.lib()


def test_every_taken_shape_divides_evenly(lib):
    rng = random.Random(7)
    taken = 0
    for _ in range(20000):
        m, mode = rng.choice([1, 16, 17, 32, 33, 64, 65, 128, 129, 256, 257, rng.randint(1, 300)]), rng.choice([1, 2])
        n = rng.choice([16, 8]) * rng.choice([rng.randint(1, 3300), 16 * rng.randint(1, 200)])
        k = rng.choice([32, 64, 128]) * rng.randint(1, 200)
        p = lib.xv_stream_gemm_parts(m, n, k, mode)
        if p == 0:
            continue
        taken += 1
        ks = 128 if m <= 64 else 64
        assert m <= 256 and n % 16 == 0 and p in (1, 2, 4, 8) and k % (p * ks) == 0, (m, n, k, mode, p)
        tiles = n // 16
        if mode == 2:
            assert p == 1 and tiles % 2 == 0
            if m <= 16:
                continue  # blocks of two tiles, any number of them
        sizes = [b for b in (1, 2, 4, 5, 6, 8, 10) if tiles % b == 0 and (224 if mode == 1 else 192) <= tiles // b * p <= 256 and (mode == 1 or b % 2 == 0)]
        assert sizes, (m, n, k, mode, p)
    assert taken > 300


def test_decoder_shapes_are_taken(lib):
    for hidden, q, kv, inter in ((1024, 2048, 1024, 3072), (4096, 4096, 1024, 12288), (5120, 8192, 1024, 25600)):
        for m in (1, 16, 17, 64, 65, 200, 256):
            assert lib.xv_stream_gemm_parts(m, hidden, inter, 1) > 0
            assert lib.xv_stream_gemm_parts(m, hidden, q, 1) > 0
            # gate/up: 3200 tiles do not divide over the CUs above 16 rows
            assert (lib.xv_stream_gemm_parts(m, 2 * inter, hidden, 2) > 0) == (m <= 16 or inter != 25600)


def test_rejects_bad_arguments(lib):
    def call(**kw):
        a = dict(x=A, xs=4096, w=A, ws=4096, out=A, os=4096, ps=64 * 4096, m=64, n=4096, k=4096, mode=1, p=4)
        a.update(kw)
        return lib.xv_stream_gemm(a["x"], a["xs"], a["w"], a["ws"], a["out"], a["os"], a["ps"], a["m"], a["n"], a["k"],
                                  a["mode"], a["p"], None)

    assert lib.xv_stream_gemm_parts(64, 4096, 4096, 1) == 4
    for kw in (dict(m=0), dict(m=257), dict(n=4096 + 16), dict(n=4090), dict(k=4096 + 8), dict(mode=0), dict(mode=3),
               dict(p=2), dict(p=8), dict(x=A + 2), dict(w=A + 8), dict(xs=4100), dict(xs=2048), dict(ws=4088), dict(ws=2048),
               dict(os=4094), dict(os=2048), dict(out=A + 8), dict(ps=64 * 4096 - 4), dict(ps=64 * 4096 + 2),
               dict(mode=2, p=1, n=24576, os=12286), dict(mode=2, p=1, n=24576, os=12288, out=A + 4),
               dict(mode=2, p=4, n=24576, os=12288)):
        assert call(**kw) == INVALID, kw


def test_operand_choice_off_the_gpu():
    from xvllm.layers.linear import GEMM_PARTS, stream_operand

    x, w = torch.zeros(4, 2048, dtype=torch.bfloat16), torch.zeros(1024, 2048, dtype=torch.bfloat16)
    assert stream_operand(x, w, None, GEMM_PARTS) is None


def test_fake_shapes():
    from torch._subclasses.fake_tensor import FakeTensorMode

    from xvllm.layers.linear import GEMM_PARTS, GEMM_SILU_MUL

    with FakeTensorMode():
        x, w = torch.empty(5, 1024, dtype=torch.bfloat16), torch.empty(6144, 1024, dtype=torch.bfloat16)
        parts = torch.ops.xv.stream_gemm(x, w, GEMM_PARTS, 2)
        act = torch.ops.xv.stream_gemm(x, w, GEMM_SILU_MUL, 1)
    assert parts.shape == (2, 5, 6144) and parts.dtype == torch.float32
    assert act.shape == (5, 3072) and act.dtype == torch.bfloat16


def test_long_batches_do_not_ask_the_library(monkeypatch):
    """Above 256 rows the choice falls on the row count alone: a prefill
    step's layers ask for each of their products."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    from xvllm.layers import linear

    asked = []
    monkeypatch.setattr(linear, "in_place_parts", lambda *a: asked.append(a) or 1)
    with FakeTensorMode():
        w = torch.empty(6144, 1024, dtype=torch.bfloat16, device="cuda")
        for m in (0, 1, 256, 257, 8192):
            x = torch.empty(m, 1024, dtype=torch.bfloat16, device="cuda")
            for packed in (None, w):
                for mode in (linear.GEMM_PARTS, linear.GEMM_SILU_MUL):
                    got = linear.stream_operand(x, w, packed, mode, internal=True)
                    assert (got is w) == (0 < m <= 256)
    assert {a[0] for a in asked} == {1, 256}


def test_every_picked_kernel_exists(lib):
    """Shapes of all sizes pick only kernels that stream_kernel_shapes names
    (the GPU test runs each of those), and a call of each gets as far as its
    launch: without a device that fails, and 0 would mean none was made."""
    shapes = stream_kernel_shapes(lib)
    rng = random.Random(11)
    for _ in range(40000):
        m, mode, k = rng.randint(1, 256), rng.choice([1, 2]), 64 * rng.randint(1, 400)
        n = 16 * rng.choice([rng.randint(1, 3300), 16 * rng.randint(1, 200)])
        kernel = stream_kernel(lib, m, n, k, mode)
        assert kernel is None or kernel in shapes, (m, n, k, kernel)
    assert {c for _, c, _ in shapes} == set(STREAM_CLASSES)
    if torch.cuda.is_available():  # (the addresses are not real)
        return
    for (mode, m, _), (n, k) in shapes.items():
        width = n if mode == 1 else n // 2
        rc = lib.xv_stream_gemm(A, k, A, k, A, width, m * n, m, n, k, mode, lib.xv_stream_gemm_parts(m, n, k, mode), None)
        assert rc not in (0, INVALID), (mode, m, n, k, rc)


def test_packing_does_not_hold_weights_read_in_place():
    """pack() keeps nothing of a weight that streams in place: replacing the
    parameter frees it, and the operand is the new one."""
    import gc
    import weakref

    import numpy as np
    from xvllm.config import Qwen3Shape
    from xvllm.models.qwen3 import Qwen3DecoderLayer

    layer = Qwen3DecoderLayer(Qwen3Shape(1024, 16, 8, 128, 3072, 1, max_position_embeddings=64), 0).to(torch.bfloat16)
    for module, name, operand in ((layer.mlp, "gate_up_proj", lambda: layer.mlp.packed[0]),
                                  (layer.mlp, "down_proj", lambda: layer.mlp.packed[1]),
                                  (layer.self_attn, "o_proj", lambda: layer.self_attn.packed_o)):
        shape = getattr(module, name).shape
        store = np.zeros(shape.numel(), np.int16)
        freed = weakref.ref(store)
        setattr(module, name, torch.nn.Parameter(torch.from_numpy(store).view(torch.bfloat16).view(shape), requires_grad=False))
        del store
        module.pack()
        assert operand().data_ptr() == getattr(module, name).data_ptr() and freed() is not None
        setattr(module, name, torch.nn.Parameter(torch.zeros(shape, dtype=torch.bfloat16), requires_grad=False))
        gc.collect()
        assert freed() is None, name
        assert operand().data_ptr() == getattr(module, name).data_ptr()
        module.pack(False)
    assert layer.mlp.packed is None and layer.self_attn.packed_o is None
