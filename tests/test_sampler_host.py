"""Sizes of the sampler's workspace (xv_sampler_workspace_size), on the CPU."""
import pytest

TOP_LIST, SEG_IDS = 64, 8192  # candidates per segment list, ids per segment of a large batch


@pytest.fixture(scope="module")
def lib():
    from xvllm import _C

    return _C.lib()


@pytest.mark.parametrize("vocab", [8192, 32000, 50257, 128256, 151936, 262144])
def test_top_k_lists_of_large_batches_fit(lib, vocab):
    """The sampled region of a large batch holds the 8-byte candidate lists of
    77936 / R rows, R segments each: 4101 rows of 151936 ids."""
    r = -(-vocab // SEG_IDS)
    rows = min(77936 // r, 65535)
    assert vocab != 151936 or rows == 4101
    greedy = -(-rows * 128 // 256) * 256
    assert lib.xv_sampler_workspace_size(rows, vocab) - greedy >= rows * r * TOP_LIST * 8


def test_size_never_decreases_with_the_batch(lib):
    for vocab in (1, 2048, 32000, 151936, 262144, 1 << 21):
        sizes = [lib.xv_sampler_workspace_size(b, vocab) for b in (*range(1, 80), 128, 129, 255, 256, 511, 512, 513, 4101)]
        assert sizes == sorted(sizes)
