"""The in-place streaming GEMM (xv_stream_gemm) against a float64 product of
the same bf16 operands, at the edges of its row classes (16, 32, 64, 128, 256
rows): the decoder's shapes, then every kernel the rule picks (row class, tile
count, form) over several turns of its ring.  Partial sums: the fp32 sum of K
products in any order is within K 2^-24 sum |x w| of the exact one.
SiLU-and-mul: at small K rtol/atol 2e-2 over the bf16-rounded products as the
packed kernel's test, and over the rings' turns the bound its roundings give."""
import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = [1, 15, 16, 17, 32, 33, 64, 65, 128, 129, 200, 256]
# (n, k): the tiles per workgroup are 1, 2 / 1, 2 / 1, 2 / 4, 8 / 5, 10 / 6 over the row classes
SHAPES = [(1024, 2048), (1024, 3072), (4096, 1024), (4096, 12288), (5120, 25600), (6144, 4096)]


def _operands(dev, m, n, k, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn((m, k), generator=g, device=dev).to(torch.bfloat16)
    w = (torch.randn((n, k), generator=g, device=dev) * 0.02).to(torch.bfloat16)
    return x, w


def _check_parts(ps, x, w):
    xd, wd = x.double(), w.double()
    want, bound = xd @ wd.T, (xd.abs() @ wd.abs().T) * (x.shape[1] * 2.0**-24)
    err = (ps.parts.double().sum(0) - want).abs() - bound
    assert torch.isfinite(ps.parts).all()
    assert (err <= 0).all(), f"max excess {err.max().item():.3g}"


@pytest.mark.parametrize("shape", SHAPES)
def test_parts(dev, shape):
    from xvllm.layers.linear import GEMM_PARTS, PartialSums, in_place_parts, streamed_into_norm

    n, k = shape
    for m in ROWS:
        p = in_place_parts(m, n, k, GEMM_PARTS)
        print(f"stream gemm m {m} n {n} k {k} parts {p}", flush=True)
        x, w = _operands(dev, m, n, k, m + n)
        ps = streamed_into_norm(x, w)
        assert isinstance(ps, PartialSums) and ps.parts.shape == (p, m, n)
        _check_parts(ps, x, w)


# blocks of 2 tiles, 4, 6 and 8 above 16 rows
@pytest.mark.parametrize("inter", [3072, 4096 * 2, 12288, 16384])
def test_silu_mul(dev, inter):
    from xvllm.layers.linear import streamed_silu_mul

    k = 512
    for m in ROWS:
        print(f"stream gemm silu m {m} I {inter}", flush=True)
        x, w = _operands(dev, m, 2 * inter, k, m + inter)
        gu = (x.double() @ w.double().T).to(torch.bfloat16).double()
        g, u = gu[:, :inter], gu[:, inter:]
        want = g * torch.sigmoid(g) * u
        out = streamed_silu_mul(x, w)
        assert out.shape == (m, inter) and out.dtype == torch.bfloat16
        err = (out.double() - want).abs() - (2e-2 + 2e-2 * want.abs())
        assert torch.isfinite(out).all() and (err <= 0).all(), f"max excess {err.max().item():.3g}"


def _silu_bound(x, w, inter):
    """The exact silu(g) u and what its roundings may move it by: the fp32 sums
    and the bf16 rounding (half of a last place, 2^-8 of the value) of g and u, that of the result, and 2^-18 for
    the fp32 exponential, reciprocal and products between; |silu'| < 1.1."""
    xd, wd = x.double(), w.double()
    gu, mass = xd @ wd.T, xd.abs() @ wd.abs().T
    d = mass * (x.shape[1] * 2.0**-24)
    d += (gu.abs() + d) * 2.0**-8
    g, u, dg, du = gu[:, :inter], gu[:, inter:], d[:, :inter], d[:, inter:]
    silu = g * torch.sigmoid(g)
    want = silu * u
    bound = 1.1 * dg * (u.abs() + du) + silu.abs() * du
    return want, bound + (want.abs() + bound) * (2.0**-8 + 2.0**-18) + 2.0**-133  # (subnormal results)


@pytest.mark.parametrize("rows", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("mode", [1, 2])
def test_every_kernel_over_turns_of_its_ring(dev, mode, rows):
    """Each kernel of the row class, at the class's fewest and most rows, over
    an odd number of stages past two turns of the deepest ring."""
    from helpers import stream_kernel, stream_kernel_shapes
    from xvllm import _C
    from xvllm.layers.linear import streamed_into_norm, streamed_silu_mul

    shapes = {k: v for k, v in stream_kernel_shapes(_C.lib()).items() if k[:2] == (mode, rows)}
    assert shapes
    for kernel, (n, k) in sorted(shapes.items()):
        for m in (rows // 2 + 1 if rows > 16 else 1, rows):
            assert stream_kernel(_C.lib(), m, n, k, mode) == kernel
            print(f"stream gemm kernel {kernel} m {m} n {n} k {k}", flush=True)
            x, w = _operands(dev, m, n, k, m + n)
            if mode == 1:
                _check_parts(streamed_into_norm(x, w), x, w)
            else:
                want, bound = _silu_bound(x, w, n // 2)
                err = (streamed_silu_mul(x, w).double() - want).abs() - bound
                assert (err <= 0).all(), f"max excess {err.max().item():.3g}"


def test_strided_rows(dev):
    """x and w as row-strided views, and x off its 16-byte alignment (copied first)."""
    from xvllm.layers.linear import streamed_into_norm

    x, w = _operands(dev, 40, 1024, 2048, 3)
    wide_x = torch.full((40, 2048 + 64), float("nan"), dtype=torch.bfloat16, device=dev)
    wide_w = torch.full((1024, 2048 + 128), float("nan"), dtype=torch.bfloat16, device=dev)
    for off in (8, 32, 3):
        wide_x[:, off : off + 2048] = x
        wide_w[:, 64 : 64 + 2048] = w
        _check_parts(streamed_into_norm(wide_x[:, off : off + 2048], wide_w[:, 64 : 64 + 2048]), x, w)


def test_rows_are_independent(dev):
    """Rows of infinities and NaN, and the row count itself, leave the other rows' bits alone."""
    from xvllm.layers.linear import streamed_into_norm

    x, w = _operands(dev, 64, 1024, 2048, 4)
    ref = streamed_into_norm(x, w).parts
    bad = x.clone()
    bad[7], bad[40, 5] = float("nan"), float("inf")
    got = streamed_into_norm(bad, w).parts
    keep = [i for i in range(64) if i not in (7, 40)]
    assert torch.equal(got[:, keep], ref[:, keep])
    assert torch.isnan(got[:, 7]).all()
    assert torch.equal(streamed_into_norm(x[:50], w).parts, ref[:, :50])


@pytest.mark.parametrize("m", [1, 40, 64, 100, 256, 257])
@pytest.mark.parametrize("width", ["0.6B", "8B"])
def test_mlp_streams_and_matches_the_library(dev, m, width):
    """The MLP, packed or not: packed models stream up to 256 rows, others the
    products into a norm where linear_into_norm splits, all within the
    bf16 tolerance of the library's product, with gradients on too (what
    those calls run on is test_gradients_keep_the_library's)."""
    from xvllm.config import QWEN3_0_6B, QWEN3_8B
    from xvllm.layers.linear import PartialSums, split_factor
    from xvllm.models.qwen3 import Qwen3MLP

    s = QWEN3_0_6B if width == "0.6B" else QWEN3_8B
    g = torch.Generator(device=dev).manual_seed(m)
    with torch.device(dev):
        mlp = Qwen3MLP(s.hidden_size, s.intermediate_size).to(torch.bfloat16)
    with torch.no_grad():
        for p in mlp.parameters():
            p.normal_(0.0, 0.02, generator=g)
        x = torch.randn((m, s.hidden_size), generator=g, device=dev).to(torch.bfloat16)
        mlp.split_k = False
        want = mlp(x).double()
        mlp.split_k = True
        split = split_factor(m, s.hidden_size, s.intermediate_size) > 1
        outs = [mlp(x)]
        assert isinstance(outs[0], PartialSums) == split
        mlp.pack()
        outs.append(mlp(x))
        assert isinstance(outs[1], PartialSums) == (m <= 256)
        mlp.pack(False)
    library = mlp(x)  # gradients of the weights asked for
    assert isinstance(library, PartialSums) == split
    outs.append(library)
    for out in outs:
        got = (out.materialize() if isinstance(out, PartialSums) else out).double()
        rel = (got - want).norm() / want.norm()
        assert rel < 1e-2, f"relative L2 {rel:.3g}"


@pytest.mark.parametrize("m", [8, 40, 100])
def test_layouts_the_library_takes(dev, m):
    """x whose rows are expanded or overlap, and weights that are expanded,
    overlap or start off a 16-byte boundary, give the library's product."""
    import torch.nn.functional as F

    from xvllm.layers.linear import PartialSums
    from xvllm.models.qwen3 import Qwen3MLP

    h, inter = 1024, 3072
    g = torch.Generator(device=dev).manual_seed(m)

    def randn(*shape, std=1.0):
        return (torch.randn(shape, generator=g, device=dev) * std).to(torch.bfloat16)

    flat = randn(8 * m + h)
    off = torch.from_dlpack(randn(2 * inter * h + 3, std=0.02)[3:])  # a storage of its own, off by 6 bytes
    assert off.storage_offset() == 0 and off.data_ptr() % 16
    weights = {"plain": randn(2 * inter, h, std=0.02), "expanded": randn(1, h, std=0.02).expand(2 * inter, h),
               "overlapping": randn(2 * inter * 8 + h, std=0.02).as_strided((2 * inter, h), (8, 1)),
               "off": off.view(2 * inter, h)}
    with torch.device(dev):
        mlp = Qwen3MLP(h, inter).to(torch.bfloat16)
    with torch.no_grad():
        mlp.down_proj.copy_(randn(h, inter, std=0.02))
        for name, w in weights.items():
            mlp.gate_up_proj = torch.nn.Parameter(w, requires_grad=False)
            for x in (randn(m, h), randn(1, h).expand(m, h), flat.as_strided((m, h), (8, 1)), randn(h, m).t()):
                print(f"layouts m {m} w {name} x stride {tuple(x.stride())}", flush=True)
                out = mlp(x)
                out = out.materialize() if isinstance(out, PartialSums) else out
                gu = F.linear(x.contiguous(), w.contiguous()).double()
                act = (gu[:, :inter] * torch.sigmoid(gu[:, :inter]) * gu[:, inter:]).to(torch.bfloat16)
                want = F.linear(act, mlp.down_proj)
                # both sides round g, u, the activation and the product to bf16: 2^-8 each
                rel = (out.double() - want.double()).norm() / want.double().norm()
                assert rel < 4 * 2.0**-8, (name, tuple(x.stride()), rel.item())


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("m", [8, 100, 300])
def test_compiles_as_one_graph(dev, m, packed):
    """torch.compile traces the MLP without a break at every row count, onto
    the library's products (Qwen3-0.6B, whose products the library does not split)."""
    from xvllm.models.qwen3 import Qwen3MLP

    g = torch.Generator(device=dev).manual_seed(m)
    with torch.device(dev):
        mlp = Qwen3MLP(1024, 3072).to(torch.bfloat16)
    with torch.no_grad():
        for p in mlp.parameters():
            p.normal_(0.0, 0.02, generator=g)
        x = torch.randn((m, 1024), generator=g, device=dev).to(torch.bfloat16)
        mlp.split_k = False
        want = mlp(x)
        mlp.split_k = True
        if packed and m > 64:  # (a packed model's shorter batches check their weights, which no trace holds)
            mlp.pack()
        torch._dynamo.reset()
        got = torch.compile(mlp, backend="eager", fullgraph=True)(x)
    assert torch.equal(got, want)


@pytest.mark.parametrize("m,packed", [(8, False), (64, False), (100, False), (100, True), (256, True)])
def test_gradients_keep_the_library(dev, m, packed):
    """With gradients on, an unpacked MLP's products and a packed one's above
    64 rows carry them (Qwen3-0.6B, whose products the library does not split;
    silu_and_mul has no backward, so gate_up is frozen)."""
    from xvllm.layers.linear import GEMM_PARTS, stream_operand
    from xvllm.models.qwen3 import Qwen3MLP

    g = torch.Generator(device=dev).manual_seed(m)
    with torch.device(dev):
        mlp = Qwen3MLP(1024, 3072).to(torch.bfloat16)
    mlp.gate_up_proj.requires_grad_(False)
    with torch.no_grad():
        for p in mlp.parameters():
            p.normal_(0.0, 0.02, generator=g)
    x = torch.randn((m, 1024), generator=g, device=dev).to(torch.bfloat16)
    go = torch.randn((m, 1024), generator=g, device=dev).to(torch.bfloat16)
    mlp.split_k = False
    want, = torch.autograd.grad(mlp(x), mlp.down_proj, go)
    mlp.split_k = True
    mlp.pack(packed)
    out = mlp(x)
    assert isinstance(out, torch.Tensor) and out.requires_grad
    got, = torch.autograd.grad(out, mlp.down_proj, go)
    # gate_up streams, so the activation behind the gradient is one bf16 rounding apart
    assert ((got.double() - want.double()).norm() / want.double().norm()).item() < 2 * 2.0**-8
    # the decode step's qkv product, which stays internal to its layer
    w = torch.nn.Parameter(torch.randn((4096, 1024), generator=g, device=dev).to(torch.bfloat16))
    assert stream_operand(x, w, None, GEMM_PARTS, internal=True) is None
    assert stream_operand(x.clone().requires_grad_(), w.detach(), None, GEMM_PARTS, internal=True) is None
    with torch.no_grad():
        assert stream_operand(x, w, None, GEMM_PARTS, internal=True) is w
