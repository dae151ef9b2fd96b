"""The successor array after a whole job: home copies of crossing k-mers hold
their duplicates' edges, however the job ran."""
import numpy as np
import pytest

import unitigcoarsening_amd as uc

pytestmark = pytest.mark.gpu


def circle(rng, length, k):
    s = "".join("ACGT"[i] for i in rng.randint(0, 4, length))
    s += s[:k - 1]
    return [s[i:i + k] for i in range(length)]


@pytest.mark.parametrize("k,l", [(31, 9), (63, 11)])
@pytest.mark.parametrize("cycles", [False, True])
def test_succ_after_a_whole_job(k, l, cycles):
    rng = np.random.RandomState(k)
    strs = set(uc.decode(uc.medium_model(9, 4_000, k), k))
    rings = [circle(rng, n, k) for n in (80, 300)] if cycles else []
    for r in rings:
        strs.update(r)
    strs = sorted(strs)
    with uc.Compactor(n_buckets=8, keep_src=True, fine_slots=64) as c:
        c.compact(uc.encode(strs, k), k, l)
        _, src, flags, _, _ = c.bucket_arrays()
        n_cycles = c.coarsen_info().n_cycles
        first, again = c.succ(), c.succ()
    assert np.array_equal(first, again) and n_cycles == len(rings)
    by_pre, n_suf = {}, {}
    for i, s in enumerate(strs):
        by_pre.setdefault(s[:-1], []).append(i)
        n_suf[s[1:]] = n_suf.get(s[1:], 0) + 1
    cut = {min(r) for r in rings}  # a ring loses the edge into its smallest k-mer
    home = {int(src[s]): s for s in range(len(src)) if flags[s] != uc.F_BORROW}
    assert len(home) == len(strs) and (flags == uc.F_LENT).any()
    for i, s in enumerate(strs):
        v = by_pre.get(s[1:], [])
        kept = len(v) == 1 and n_suf[s[1:]] == 1 and strs[v[0]] not in cut
        assert first[home[i]] == (home[v[0]] if kept else 0xFFFFFFFF), (i, s)
