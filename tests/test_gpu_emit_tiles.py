"""Emission and contraction tiles of every size: the tile grows with the
job's slots (64 slots up to 131 072, then 128, 256 and 512), and a tile's text
goes through LDS when 64 heads' lines fit and straight to memory when not."""
import random

import numpy as np
import pytest

import oracle
import unitigcoarsening_amd as uc

pytestmark = pytest.mark.gpu


def path_kmers(rng, length, k):
    s = "".join(rng.choice("ACGT") for _ in range(length))
    return sorted({s[i:i + k] for i in range(length - k + 1)})


@pytest.mark.parametrize("k", [3, 31, 32, 33, 63, 64])
@pytest.mark.parametrize("genome", [70, 4_000, 116_000, 122_000, 232_000, 245_000, 470_000, 490_000])
def test_text_at_the_tile_sizes(k, genome):
    # (the tile boundaries fall at 118-123 k, 236-246 k and 472-490 k k-mers here)
    kmers = uc.medium_model(genome + k, genome, k)
    want, _, _ = oracle.textbook(kmers, k)
    with uc.Compactor(n_buckets=16) as c:
        got = c.compact(kmers, k, min(9, k - 1))
    assert uc.sorted_lines(got) == uc.sorted_lines(want)


@pytest.mark.parametrize("k", [31, 63])
def test_long_and_short_lines_in_one_tile(k):
    # one bucket: lines of 1 to 4000 k-mers side by side, some too long for the stage
    rng = random.Random(5)
    strs = set()
    for n in [1] * 300 + [2] * 50 + [5, 17, 40, 200, 4000]:
        strs.update(path_kmers(rng, n + k - 1, k))
    kmers = uc.encode(sorted(strs), k)
    want, _, _ = oracle.textbook(kmers, k)
    for B in (1, 8):
        with uc.Compactor(n_buckets=B, sample_log2=4) as c:
            assert uc.sorted_lines(c.compact(kmers, k, 7)) == uc.sorted_lines(want)
    idx = np.random.RandomState(1).permutation(kmers.shape[0])
    with uc.Compactor(n_buckets=4) as c:
        assert uc.sorted_lines(c.compact(kmers[idx], k, 7)) == uc.sorted_lines(want)
