"""The sampled path by per-key counts, where its cases change: logits below,
at the edges of and past the counted magnitudes, zeros, masked rows, heavy
ties, and vocabularies around its segment cuts.  Ids equal the C oracle's."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


def rows(kind, b, v, rng):
    x = rng.standard_normal((b, v)).astype(np.float32) * 2
    if kind == "tiny":  # a few magnitudes in (0, 2^-22), listed beside the counts
        x[:, rng.integers(0, v, 40)] *= 1e-8
    elif kind == "many_tiny":  # more than a segment's list holds
        x[:, ::2] *= 1e-8
    elif kind == "zero_cut":  # the cut falls among exact zeros of both signs
        x = np.where(rng.random((b, v)) < 0.9, np.float32(0), np.abs(x))
        x[:, ::3] *= -1
    elif kind == "all_negative":  # the maximum lies in the negative half
        x = -np.abs(x) - 0.25
    elif kind == "max_zero":
        x = -np.abs(x)
        x[:, v // 2] = 0
    elif kind == "edges":  # both ends of the counted magnitudes
        x[:, 1 % v] = 1020.0
        x[:, 2 % v] = 2.0 ** -22
        x[:, 3 % v] = -1020.0
    elif kind == "past_top":
        x[:, 5 % v] = 1024.0
    elif kind == "masked":  # most ids masked, as constrained decoding leaves them
        x[rng.random((b, v)) < 0.95] = -np.inf
        x[:, 0] = 1.0
        x[b // 2:][np.isinf(x[b // 2:])] = np.finfo(np.float32).min
    elif kind == "hot_far":  # -2^10 and below with mass: a temperature of 1e4
        x *= 600
    elif kind == "massive":  # thousands of ids on one key
        x = np.round(x)
    elif kind == "one_value":
        x[:] = 3.5
    return x


@pytest.mark.parametrize("kind", ["tiny", "many_tiny", "zero_cut", "all_negative", "max_zero", "edges", "past_top",
                                  "masked", "hot_far", "massive", "one_value"])
@pytest.mark.parametrize("v", [2048, 16391, 65537])
def test_count_path_matches_the_oracle(dev, kind, v):
    import oracle.sampler as S
    from xvllm.sampler import sample

    rng = np.random.default_rng(v + len(kind))
    b = 12
    logits = torch.from_numpy(rows(kind, b, v, rng)).to(torch.bfloat16)
    temps = torch.full((b,), 1e4 if kind == "hot_far" else 0.9)
    u = torch.from_numpy(rng.random(b).astype(np.float32))
    tps = torch.from_numpy(rng.uniform(0.2, 1.0, b).astype(np.float32))
    tks = torch.from_numpy(rng.integers(1, v, b).astype(np.int32))
    mps = torch.from_numpy((10.0 ** rng.uniform(-14, -0.1, b)).astype(np.float32))
    bits = logits.view(torch.int16).numpy().view(np.uint16)
    g = [t.to(dev) for t in (logits, temps, tps, tks, mps, u)]
    for flags in (0, 2, 4, 8, 2 | 4 | 8):
        want = S.sample(bits, temps.numpy(), tps.numpy(), tks.numpy(), mps.numpy(), u.numpy(), flags)
        got = sample(*g, use_top_k=bool(flags & 2), use_top_p=bool(flags & 4), use_min_p=bool(flags & 8))
        assert np.array_equal(got.cpu().numpy(), want), (flags, got.cpu().numpy(), want)


def near_zero(kind, b, v, rng):
    """Rows whose largest logits, and so their cuts, lie at zero."""
    x = rng.standard_normal((b, v)).astype(np.float32) * 2
    x -= x.max(1, keepdims=True)  # "shifted": each row's maximum is 0
    if kind == "log_probs":  # of a row with one likely id
        x[:, v // 3] = 25.0
        x -= np.log(np.exp(x.astype(np.float64)).sum(1, keepdims=True)).astype(np.float32)
    elif kind == "zeros":
        x[rng.random((b, v)) < 0.7] = 0
        x[rng.random((b, v)) < 0.2] *= -1
    elif kind == "all_zero":
        x[:] = np.where(rng.random((b, v)) < 0.5, np.float32(0), np.float32(-0.0))
    elif kind in ("listed", "listed_flat"):  # values of both signs listed beside the counts, repeated ones, zeros between
        x = np.minimum(x, -0.5 if kind == "listed" else -8.0)
        for row in x:
            ids = rng.permutation(v)[: min(v, 80)]
            row[ids[:56]] = rng.choice(rng.choice([-1, 1], 30) * 2.0 ** -rng.uniform(22.1, 120, 30), ids[:56].size)
            row[ids[56:68]] = 0
            row[ids[68:]] = -0.0
    elif kind == "listed_hot":  # their masses differ: read at a temperature of 1e-5 or so
        x = np.minimum(x, -0.5)
        x[:, rng.permutation(v)[:40]] = rng.uniform(-2e-7, 2e-7, (b, min(v, 40)))
    elif kind == "one_mass":  # more small values than any list takes, a maximum that makes them equal
        x[:, ::2] *= 1e-8
        x[:, v // 2] = 9.0
    elif kind == "nearly_one_mass":  # a maximum at which the small values' distances just differ
        x[:, ::2] = rng.uniform(-2.3e-7, 2.3e-7, x[:, ::2].shape)
        x[:, 1::2] = np.minimum(x[:, 1::2], -1)
        x[:, v // 2] = rng.choice([1.0, 2.0, 3.99, 4.0, 5.0, 7.99], b)
    elif kind == "too_many":  # more listed values than one row's list takes
        x = np.minimum(x, -0.5)
        x[:, ::7] = rng.uniform(-2e-7, 2e-7, x[:, ::7].shape)
    return x


@pytest.mark.parametrize("kind", ["shifted", "log_probs", "zeros", "all_zero", "listed", "listed_flat", "listed_hot",
                                  "one_mass", "nearly_one_mass", "too_many"])
@pytest.mark.parametrize("v", [33, 2048, 16391, 65537])
def test_cuts_at_zero_match_the_oracle(dev, kind, v):
    import oracle.sampler as S
    from xvllm.sampler import sample

    rng = np.random.default_rng(v + len(kind))
    b = 24
    logits = torch.from_numpy(near_zero(kind, b, v, rng).astype(np.float32)).to(torch.bfloat16)
    temps = torch.full((b,), 1.2e-5 if kind == "listed_hot" else 0.9)
    u = torch.from_numpy(rng.random(b).astype(np.float32))
    tps = torch.from_numpy(rng.uniform(0.02, 1.0, b).astype(np.float32))
    tks = torch.from_numpy(rng.integers(1, min(v, 100), b).astype(np.int32))  # ranks among the listed values and zeros
    tks[::3] = torch.from_numpy(rng.integers(1, v, tks[::3].numel()).astype(np.int32))
    mps = torch.from_numpy((10.0 ** rng.uniform(-6, -0.1, b)).astype(np.float32))
    mps[::4] = 1.0
    bits = logits.view(torch.int16).numpy().view(np.uint16)
    g = [t.to(dev) for t in (logits, temps, tps, tks, mps, u)]
    for flags in (0, 2, 4, 8, 2 | 4, 2 | 4 | 8):
        want = S.sample(bits, temps.numpy(), tps.numpy(), tks.numpy(), mps.numpy(), u.numpy(), flags)
        got = sample(*g, use_top_k=bool(flags & 2), use_top_p=bool(flags & 4), use_min_p=bool(flags & 8))
        assert np.array_equal(got.cpu().numpy(), want), (flags, got.cpu().numpy(), want)


def call_us(logits, **kw):
    """Time of a sampled call inside a graph of 20, the fastest of 7."""
    from xvllm.sampler import reserve_workspace, sample

    b, v = logits.shape
    reserve_workspace(logits.device, b, v)
    temps, u = torch.ones(b, device=logits.device), torch.full((b,), 0.37, device=logits.device)
    sample(logits, temps, uniforms=u, **kw)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for _ in range(20):
            sample(logits, temps, uniforms=u, **kw)
    best = 1e30
    for _ in range(7):
        e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        e[0].record()
        graph.replay()
        e[1].record()
        e[1].synchronize()
        best = min(best, e[0].elapsed_time(e[1]) * 50)
    return best


def usual_and(dev, make, b=32, v=151936):
    """Logits N(0, 2) and make(them), on the device."""
    g = torch.Generator(device=dev).manual_seed(3)
    x = torch.randn((b, v), generator=g, device=dev) * 2
    return x.to(torch.bfloat16), make(x.clone()).to(torch.bfloat16)


def no_slower(dev, make, modes, most):
    """Calls on make(usual logits) take at most `most` times those on usual
    ones: the counts settle the rows.  A row left to the one-workgroup path
    takes four times as long and more."""
    usual, rows = usual_and(dev, make)
    b = usual.shape[0]
    args = {"plain": {}, "top_p": dict(top_ps=torch.full((b,), 0.95, device=dev), use_top_p=True),
            "top_k": dict(top_ks=torch.full((b,), 50, dtype=torch.int32, device=dev), use_top_k=True),
            "min_p": dict(min_ps=torch.full((b,), 0.05, device=dev), use_min_p=True)}
    for mode in modes:
        a, c = call_us(usual, **args[mode]), call_us(rows, **args[mode])
        assert c <= most * a, f"{mode}: {c:.1f} us, usual rows {a:.1f}"


@pytest.mark.parametrize("kind", ["shifted", "log_probs", "max_zero", "all_zero"])
def test_rows_near_zero_are_settled_by_the_counts(dev, kind):
    def make(x):
        if kind == "log_probs":
            x[:, 7] = 30.0
            return torch.log_softmax(x, -1)
        if kind == "max_zero":
            x = -x.abs()
            x[:, 7] = 0
            return x
        return torch.zeros_like(x) if kind == "all_zero" else x - x.amax(1, keepdim=True)

    no_slower(dev, make, ["plain", "top_p", "top_k", "min_p"], 2.5 if kind == "all_zero" else 1.5)


@pytest.mark.parametrize("modes", ["plain", "top_k", "min_p"])
def test_many_small_values_are_settled_by_the_counts(dev, modes):
    """Half of a row's ids below 2^-22, of one mass beside a maximum of 8 and
    more (calls whose cut lies among them excepted)."""
    def make(x):
        x[:, ::2] *= 1e-8
        return x

    no_slower(dev, make, [modes], 1.9)


def large(kind, b, v, rng):
    """Rows with logits of 2^10 and above."""
    x = rng.standard_normal((b, v)).astype(np.float32) * 2
    few = min(v, 30)
    ids = np.stack([rng.permutation(v)[:few] for _ in range(b)])
    if kind == "one":
        x[:, v // 3] = 1500
    elif kind == "some":  # a few within reach of each other, repeated values
        np.put_along_axis(x, ids, (rng.integers(150, 154, (b, few)) * 8).astype(np.float32), 1)
    elif kind == "around":  # the cut on either side of 2^10, and in mid or far with them
        x = x * 5 + 1010
        np.put_along_axis(x, ids, rng.choice([0.0, -0.0, 1e-8, -1e5], (b, few)).astype(np.float32), 1)
        x[:, few + 5:] = np.minimum(x[:, few + 5:], 1020)  # few of them at or past it
    elif kind == "spread":  # a third of the row
        x *= 600
    elif kind == "level":  # more of them with mass than a list holds
        x += 2000
    elif kind == "top_far":  # everything past the counted magnitudes
        x = np.where(x > 4, np.float32(3000), np.float32(-3000)) + x
    elif kind == "huge":  # scaled past 2^20
        x = np.exp2(x * 10 + 25)
    return x


@pytest.mark.parametrize("kind", ["one", "some", "around", "spread", "level", "top_far", "huge"])
@pytest.mark.parametrize("v", [33, 2048, 16391, 65537])
@pytest.mark.parametrize("t", [0.9, 20.0])
def test_large_logits_match_the_oracle(dev, kind, v, t):
    import oracle.sampler as S
    from xvllm.sampler import sample

    rng = np.random.default_rng(v + len(kind))
    b = 24
    logits = torch.from_numpy(large(kind, b, v, rng).astype(np.float32)).to(torch.bfloat16)
    temps = torch.full((b,), t)
    u = torch.from_numpy(rng.random(b).astype(np.float32))
    tps = torch.from_numpy(rng.uniform(0.02, 1.0, b).astype(np.float32))
    tks = torch.from_numpy(rng.integers(1, min(v, 40), b).astype(np.int32))
    mps = torch.from_numpy((10.0 ** rng.uniform(-14, -0.1, b)).astype(np.float32))
    mps[::4] = 1.0
    bits = logits.view(torch.int16).numpy().view(np.uint16)
    g = [x.to(dev) for x in (logits, temps, tps, tks, mps, u)]
    for flags in (0, 2, 4, 8, 2 | 4, 2 | 4 | 8):
        want = S.sample(bits, temps.numpy(), tps.numpy(), tks.numpy(), mps.numpy(), u.numpy(), flags)
        got = sample(*g, use_top_k=bool(flags & 2), use_top_p=bool(flags & 4), use_min_p=bool(flags & 8))
        assert np.array_equal(got.cpu().numpy(), want), (flags, got.cpu().numpy(), want)


@pytest.mark.parametrize("kind", ["one", "spread"])
def test_rows_with_large_logits_are_settled_by_the_counts(dev, kind):
    def make(x):
        if kind == "spread":
            return x * 600
        x[:, 7] = 1500
        return x

    # two more passes over such a segment and its list: 1.6 to 1.75 times a usual row where a third of the ids are large
    no_slower(dev, make, ["plain", "top_p", "top_k", "min_p"], 2.5 if kind == "spread" else 1.5)


@pytest.mark.parametrize("v", [33, 2048, 65537])
def test_rows_without_mass_match_the_oracle(dev, v):
    """A scaled maximum that is not finite leaves no mass anywhere: +inf once
    and twice, beside NaN and -inf; -inf alone; finite values past fp32's range
    once scaled, of either sign; and rows that only look so."""
    import oracle.sampler as S
    from xvllm.sampler import sample

    rng = np.random.default_rng(v)
    x = rng.standard_normal((12, v)).astype(np.float32) * 2
    x[0, v // 2] = np.inf
    x[1, [v // 3, v - 1]] = np.inf
    x[2, :5] = [np.nan, -np.inf, np.inf, np.nan, 3e38]
    x[3] = -np.inf
    x[4] = np.where(rng.random(v) < 0.5, np.nan, -np.inf)
    x[5, 7] = 3e38
    x[6] = -3e38
    x[7] = np.where(rng.random(v) < 0.5, np.float32(-2e38), -np.inf)
    x[8] = np.nan
    x[9] = -1e5  # finite once scaled: every id alike
    x[10] = np.where(rng.random(v) < 0.9, -np.inf, np.float32(-2000))
    x[11, ::2] = -np.inf
    temps = torch.full((12,), 0.45)
    u = torch.from_numpy(rng.random(12).astype(np.float32))
    tps, mps = torch.full((12,), 0.7), torch.full((12,), 0.1)
    tks = torch.full((12,), 9, dtype=torch.int32)
    logits = torch.from_numpy(x).to(torch.bfloat16)
    bits = logits.view(torch.int16).numpy().view(np.uint16)
    g = [y.to(dev) for y in (logits, temps, tps, tks, mps, u)]
    for flags in (0, 2, 4, 8, 2 | 4 | 8):
        want = S.sample(bits, temps.numpy(), tps.numpy(), tks.numpy(), mps.numpy(), u.numpy(), flags)
        got = sample(*g, use_top_k=bool(flags & 2), use_top_p=bool(flags & 4), use_min_p=bool(flags & 8))
        assert np.array_equal(got.cpu().numpy(), want), (flags, got.cpu().numpy(), want)


@pytest.mark.parametrize("value", [float("inf"), float("-inf")])
def test_rows_without_mass_take_one_scan(dev, value):
    """The largest key is known from the counts: one more pass over the row, not two."""
    def make(x):
        x[:, 9 if value > 0 else slice(None)] = value
        return x

    no_slower(dev, make, ["plain", "top_p", "top_k", "min_p"], 1.6)
