"""The device's plans over many rows: LDS groups per coarse bucket (one wave up
to 512 fine buckets, else four) and fine-sort tiles per row (4096 rows a
round).  A batch's texts are its sets' own."""
import numpy as np
import pytest

import unitigcoarsening_amd as uc

pytestmark = pytest.mark.gpu


# (buckets, set sizes) at 64 slots per fine bucket: 512 and 1024 fine buckets per coarse bucket, beside sets of one and
# none; 4096 rows and 4352 (16 and 17 sets of 256 buckets)
@pytest.mark.parametrize("k,B,sizes", [
    (31, 1, [28_000, 500, 0, 27_000]), (31, 1, [40_000, 500, 0, 3_000]), (63, 1, [40_000, 28_000]),
    (31, 4, [112_000, 160_000, 64]), (31, 256, [70_000] * 16), (31, 256, [70_000] * 17),
])
@pytest.mark.parametrize("group_slots", [0, 256])
def test_batch_equals_its_sets(k, B, sizes, group_slots):
    sets = [uc.medium_model(200 + i, max(n + n // 16, 100), k)[:n] for i, n in enumerate(sizes)]
    with uc.Compactor(n_buckets=B, fine_slots=64, group_slots=group_slots) as c:
        texts = c.compact_sets(sets, k, 11)
        for i, (s, t) in enumerate(zip(sets, texts)):
            assert t == (c.compact(np.ascontiguousarray(s), k, 11) if s.shape[0] else b""), i
