"""The slot order of the bucketing, whatever its two passes take of the fine
bits: placements sorted by (set, coarse bucket, fine index), input order kept
inside a fine bucket, a k-mer's home copy before its borrowed one."""
import numpy as np
import pytest

import oracle
import unitigcoarsening_amd as uc

pytestmark = pytest.mark.gpu


def fine_count(n, B, fine_slots):
    want = (n * 112 // 100 + B * fine_slots - 1) // (B * fine_slots)
    s = 1
    while s < want and s < 1024:
        s *= 2
    return s


def minima(x, k, l, order):
    """Minimum order over the l-mers of every k-mer's (k-1)-prefix and (k-1)-suffix."""
    code, low, ends = np.zeros(x.shape[0], np.int64), None, []
    for i in range(k):  # (first character most significant)
        code = (code << 2 | (x[:, i // 16].astype(np.int64) >> (2 * (i % 16))) & 3) & (4 ** l - 1)
        if l <= i + 1 < k:
            o = order[code]
            ends = ends or [o]
            low = o if i + 1 == l + 1 else low if low is None else np.minimum(low, o)
    last = order[code]
    return np.minimum(ends[0], low), np.minimum(low, last)


# (k, buckets, fine_slots, set sizes): one pass with all fine bits (up to 1024 rows), two passes with the fine bits
# split or not, sets with fewer fine bits than pass 1 takes (none, some), one set, an empty set, 1 and 1024 buckets,
# rows long enough for the fine sort's long rounds (32 768 slots on average)
@pytest.mark.parametrize("k,B,fine_slots,sizes", [
    (31, 1, 64, [12_000]), (31, 1, 64, [90_000]), (31, 64, 64, [5_000]), (31, 64, 64, [60_000]), (31, 128, 64, [9_000]),
    (31, 1024, 64, [3_000]), (31, 1024, 64, [140_000]), (63, 1024, 64, [140_000]), (63, 64, 64, [60_000]),
    (31, 16, 64, [200, 9_000, 0, 2_100]), (31, 4, 64, [40, 70_000, 300, 2_500]),
    (31, 2, 64, [1_150_000]), (47, 2, 64, [1_150_000]),
])
def test_slots_are_the_stable_sort_by_fine_bucket(k, B, fine_slots, sizes):
    l, seed = 8, 77
    kmers = [uc.medium_model(3 + i, max(n + n // 16, 100), k)[:n] for i, n in enumerate(sizes)]
    sizes = [x.shape[0] for x in kmers]
    with uc.Compactor(n_buckets=B, seed=seed, keep_src=True, fine_slots=fine_slots) as c:
        c.load(np.concatenate(kmers), k, set_sizes=sizes)
        c.bucketize(l)
        rows, src, flags, ph, pb = c.bucket_arrays()
        n_fine = c.bucket_info().n_fine_buckets
    order = oracle.lmer_order_table(l, seed).astype(np.int64)
    subs = [fine_count(n, B, fine_slots) for n in sizes]
    assert n_fine == B * sum(subs)
    keys, ids, want_flags, n0 = [], [], [], 0
    for s, (x, sub) in enumerate(zip(kmers, subs)):
        fine = [o & (B * sub - 1) for o in minima(x, k, l, order)]
        slot_key = [((s * B + (f & (B - 1))) << 32) | f // B for f in fine]
        n = x.shape[0]
        cross = fine[0] != fine[1]
        keys += [slot_key[0], slot_key[1][cross]]
        ids += [2 * (n0 + np.arange(n)), 2 * (n0 + np.nonzero(cross)[0]) + 1]
        want_flags += [np.where(cross, uc.F_LENT, 0), np.full(int(cross.sum()), uc.F_BORROW)]
        n0 += n
    keys, ids, want_flags = np.concatenate(keys), np.concatenate(ids), np.concatenate(want_flags)
    at = np.lexsort((ids, keys))
    assert np.array_equal(src, ids[at] // 2)
    assert np.array_equal(flags, want_flags[at])
    G = B * len(sizes)
    assert np.array_equal(rows, np.searchsorted(keys[at] >> 32, np.arange(G + 1)))
    # the pairs, in any order: every crossing k-mer's home slot with its borrowed one
    assert np.array_equal(src[ph], src[pb])
    assert np.array_equal(np.sort(src[ph]), np.sort(ids[ids % 2 == 1] // 2))
    assert (flags[ph] == uc.F_LENT).all() and (flags[pb] == uc.F_BORROW).all()
