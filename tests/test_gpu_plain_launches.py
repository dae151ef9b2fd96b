"""The plain form finds edges bucket by bucket: every bucket's LDS groups and
hash slices are launches of its own, where the batched form takes all buckets'
in one.  The texts are the same bytes."""
import numpy as np
import pytest

import unitigcoarsening_amd as uc

pytestmark = pytest.mark.gpu


# (k, l, buckets, kernel): many small fine buckets; few minimizers, whose fine buckets are split by key hash
@pytest.mark.parametrize("k,l,B,kernel", [(31, 11, 16, "k_edge_lds"), (63, 11, 8, "k_edge_lds"), (31, 3, 2, "k_edge_slice")])
def test_a_launch_per_bucket(k, l, B, kernel):
    kmers = uc.medium_model(11, 300_000, k)
    texts, launches = [], []
    for mode in (uc.UC_MODE_BATCHED, uc.UC_MODE_PLAIN):
        with uc.Compactor(n_buckets=B, mode=mode, profile=True, keep_src=True) as c:
            texts.append(c.compact(kmers, k, l))
            launches.append(c.kernel_stats()[kernel][1])
            rows = np.diff(c.bucket_arrays()[0].astype(np.int64))
    assert texts[0] == texts[1]
    assert (rows > 0).all() and rows.shape[0] == B
    assert launches == [1, B]
