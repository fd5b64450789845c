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
