"""Scans whose tile sums are scanned in turn (more than 4096 of 2048 values):
the histogram and the group counts of a batch of 9000 sets in 1024 buckets."""
import pytest

import oracle
import unitigcoarsening_amd as uc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [31, 63])
def test_batch_of_many_small_sets(k):
    kinds = [uc.medium_model(60 + i, 12 + 9 * i, k) for i in range(8)]
    want = [uc.sorted_lines(oracle.textbook(x, k)[0]) for x in kinds]
    order = [(7 * i + i // 13) % 8 for i in range(9_000)]
    with uc.Compactor(n_buckets=1024) as c:
        texts = c.compact_sets([kinds[q] for q in order], k, 11)
    assert len(texts) == len(order)
    for i, (q, t) in enumerate(zip(order, texts)):
        assert uc.sorted_lines(t) == want[q], i
