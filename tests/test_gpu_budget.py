"""Jobs under a budget that just holds them: those below fitted these bytes
when pass-1 tiles had 2048 k-mers and contraction tiles 2048 slots, and still
do; the text is that of the same job without a budget."""
import numpy as np
import pytest

import unitigcoarsening_amd as uc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("l,B,sizes,low_memory,budget", [
    (11, 1024, [60_000], False, 8_910_000),
    (3, 1024, [800_000], False, 159_000_000),
    (3, 1024, [800_000], True, 62_600_000),
    (11, 512, [50_000] * 20, True, 77_800_000),
    (11, 1024, [400_000, 30, 0, 60_000, 9_000], True, 37_000_000),
])
def test_fits_its_budget(l, B, sizes, low_memory, budget):
    k = 31
    base = uc.medium_model(5, max(sizes) + max(sizes) // 8 + 100, k)
    sets = [base[:n] for n in sizes]
    want = None
    for bytes_ in (0, budget):
        with uc.Compactor(n_buckets=B, low_memory=low_memory, hbm_budget=bytes_) as c:
            c.load(np.concatenate(sets), k, set_sizes=[s.shape[0] for s in sets])
            c.compact_loaded(l)
            got = c.text()
            assert not bytes_ or c.timing().device_peak_bytes <= bytes_
        want = got if want is None else want
        assert got == want
