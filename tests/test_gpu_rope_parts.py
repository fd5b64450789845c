"""q/k norm + RoPE + KV store from split-K partial sums: bit-equal to the same
kernel on the bf16 sum of the partials (part 0 first, rounded once), bf16 and
fp8 caches of both page orders and block sizes, skipped slots, one to eight
parts, padded strides; bad arguments raise."""
import pytest
import torch

import xvllm.layers.ops  # noqa: F401  (registers the xv:: ops)

pytestmark = pytest.mark.gpu
D = 128


def _cache(dev, blocks, bs, hkv, hnd, dtype):
    shape = (2, blocks, hkv, bs, D) if hnd else (2, blocks, bs, hkv, D)
    c = torch.zeros(shape, device=dev, dtype=torch.bfloat16).to(dtype)
    return c.transpose(2, 3) if hnd else c


@pytest.mark.parametrize("tokens,parts,hq,hkv,bs,hnd,fp8", [
    (1, 1, 16, 8, 16, True, False), (7, 8, 16, 8, 16, False, False), (64, 4, 32, 8, 16, True, True),
    (33, 2, 64, 8, 256, True, False), (5, 3, 8, 8, 256, False, True), (200, 4, 32, 8, 16, True, False)])
def test_equals_the_store_on_the_sum(dev, tokens, parts, hq, hkv, bs, hnd, fp8):
    print(f"rope parts T {tokens} P {parts} heads {hq}/{hkv} block {bs} hnd {hnd} fp8 {fp8}", flush=True)
    g = torch.Generator(device=dev).manual_seed(tokens * 10 + parts)
    width = (hq + 2 * hkv) * D
    buf = torch.randn((parts, tokens, width + 8), generator=g, device=dev) * 0.7
    p = buf[:, :, :width]
    acc = p[0].clone()
    for i in range(1, parts):
        acc += p[i]
    qkv = acc.to(torch.bfloat16)
    qw = (1 + 0.1 * torch.randn(D, generator=g, device=dev)).to(torch.bfloat16)
    kw = (1 + 0.1 * torch.randn(D, generator=g, device=dev)).to(torch.bfloat16)
    pos = torch.randint(0, 512, (tokens,), generator=g, device=dev)
    cs = torch.randn((512, D), generator=g, device=dev)
    blocks = tokens // bs + 3
    slots = torch.randperm(blocks * bs, generator=g, device=dev)[:tokens].to(torch.int32)
    if tokens > 2:
        slots[1] = -1
    dt = torch.float8_e4m3fn if fp8 else torch.bfloat16
    ca, cb = _cache(dev, blocks, bs, hkv, hnd, dt), _cache(dev, blocks, bs, hkv, hnd, dt)
    scales = (0.03, 0.05) if fp8 else (1.0, 1.0)
    q = qkv[:, : hq * D].view(tokens, hq, D)
    k = qkv[:, hq * D : (hq + hkv) * D].view(tokens, hkv, D)
    v = qkv[:, (hq + hkv) * D :].view(tokens, hkv, D)
    want = torch.ops.xv.qk_norm_rope_store(q, k, v, qw, kw, 1e-6, pos, cs, ca[0], ca[1], slots, *scales)
    got = torch.ops.xv.qk_norm_rope_store_parts(p, hq, qw, kw, 1e-6, pos, cs, cb[0], cb[1], slots, *scales)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    assert torch.equal(ca.contiguous().view(torch.uint8), cb.contiguous().view(torch.uint8))
    assert got.abs().sum() > 0 and ca.contiguous().view(torch.uint8).any()


def test_rejects_bad_arguments(dev):
    hq, hkv = 16, 8
    ones = torch.ones(D, dtype=torch.bfloat16, device=dev)
    cache = _cache(dev, 2, 16, hkv, False, torch.bfloat16)
    pos, cs = torch.zeros(3, dtype=torch.int64, device=dev), torch.zeros((4, D), device=dev)
    slots = torch.zeros(3, dtype=torch.int32, device=dev)

    def call(parts, slots=slots, cache=cache, scale=1.0):
        return torch.ops.xv.qk_norm_rope_store_parts(parts, hq, ones, ones, 1e-6, pos, cs, cache[0], cache[1], slots,
                                                     scale, 1.0)

    good = torch.zeros((2, 3, (hq + 2 * hkv) * D), device=dev)
    call(good)
    for bad in (good.to(torch.bfloat16), good[0], good[:, :, : hq * D], good[:, :2]):
        with pytest.raises(ValueError):
            call(bad)
    with pytest.raises(RuntimeError):  # nine partials
        call(torch.zeros((9, 3, (hq + 2 * hkv) * D), device=dev))
    with pytest.raises(RuntimeError):  # a zero fp8 scale
        call(good, cache=_cache(dev, 2, 16, hkv, False, torch.float8_e4m3fn), scale=0.0)


def _decode_attention(dev, rows, slack=0, seed=0):
    """A decode call of one Qwen3Attention (1024 wide, 16 q / 8 kv heads) whose
    qkv product streams: (layer, its arguments, the pool's attention context)."""
    from xvllm.config import Qwen3Shape
    from xvllm.kv_pool import KVPool
    from xvllm.layers.attention import AttnInputs, AttnMetadata, attention_context
    from xvllm.models.qwen3 import Qwen3Attention

    cfg = Qwen3Shape(1024, 16, 8, D, 3072, 1, max_position_embeddings=1024)
    g = torch.Generator(device=dev).manual_seed(seed)
    with torch.device(dev):
        layer = Qwen3Attention(cfg, 0).to(torch.bfloat16)
    with torch.no_grad():
        layer.qkv_proj.normal_(0.0, 0.02, generator=g)
        layer.o_proj.normal_(0.0, 0.02, generator=g)
        hidden = torch.randn((rows, 1024), generator=g, device=dev).to(torch.bfloat16)
    pool = KVPool(cfg, num_blocks=4 * rows, block_size=16, device=dev, dtype=torch.bfloat16)
    pool.kv_cache.normal_(generator=g)
    lens = torch.randint(1, 64, (rows,), generator=g, device=dev, dtype=torch.int32)
    bt = torch.arange(4 * rows, dtype=torch.int32, device=dev).view(rows, 4)
    last = (lens - 1).long()
    slots = bt.gather(1, (last // 16)[:, None])[:, 0] * 16 + (last % 16).to(torch.int32)
    pad = lambda t, value: torch.cat([t, t.new_full((slack,), value)])  # noqa: E731
    attn = AttnInputs(slot_mapping=pad(slots, -1), is_prefill=False, block_tables=bt, cache_seqlens=lens)
    return layer, (pad(last, 0), hidden, attn), pool, attention_context(AttnMetadata(kv_cache=pool.kv_cache))


@pytest.mark.parametrize("rows", [3, 64])
def test_decode_takes_buffers_of_a_larger_batch(dev, rows):
    """Positions and slots longer than the batch: its own rows are read, as
    the store of the unsplit product does."""
    outs = []
    for slack in (0, 9):
        layer, args, pool, ctx = _decode_attention(dev, rows, slack)
        with torch.no_grad(), ctx:
            out = layer(*args)
        outs.append((getattr(out, "parts", out), pool.kv_cache))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("how", ["pre_hook", "hook", "global", "forward"])
def test_observers_of_attention_see_k_and_v(dev, how):
    """Hooks on the decoder's Attention, and a forward in its place, get the
    projection's k and v [T, Hkv, D], and the output does not change."""
    import torch.nn.functional as F

    rows = 5
    layer, args, _, ctx = _decode_attention(dev, rows)
    seen = []

    def see(*a):
        inputs = a if how == "forward" else a[1]
        if how != "global" or a[0] is layer.attn:
            seen.append((inputs[1], inputs[2]))

    with torch.no_grad(), ctx:
        plain = layer(*args)
        if how == "pre_hook":
            handle = layer.attn.register_forward_pre_hook(see)
        elif how == "hook":
            handle = layer.attn.register_forward_hook(see)
        elif how == "global":
            handle = torch.nn.modules.module.register_module_forward_pre_hook(see)
        else:
            own, handle = layer.attn.forward, None
            layer.attn.forward = lambda *a: (see(*a), own(*a))[1]
        out = layer(*args)
        if handle is not None:
            handle.remove()
        qkv = F.linear(args[1].double(), layer.qkv_proj.double())
    (k, v), = seen
    for got, want in ((k, qkv[:, layer.q_size : layer.q_size + layer.kv_size]), (v, qkv[:, layer.q_size + layer.kv_size :])):
        assert got.shape == (rows, layer.num_kv_heads, D) and got.dtype == torch.bfloat16
        # an fp32 sum rounded to bf16 once
        err = (got.double().reshape(rows, -1) - want).norm() / want.norm()
        assert err < 2.0**-8, err.item()
    assert torch.equal(getattr(out, "parts", out), getattr(plain, "parts", plain))
