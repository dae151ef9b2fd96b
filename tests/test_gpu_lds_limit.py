"""A device with 64 KiB of LDS per workgroup: what needs more takes the forms
that do with less, and the text is the same bytes."""
import ctypes as C

import pytest

import unitigcoarsening_amd as uc

pytestmark = pytest.mark.gpu


# 4.3 M k-mers: more tile sums than 64 KiB hold.  2.5 M in 64 buckets of 16 fine buckets: 1024 rows in one pass, whose
# counters are 74 KB.
@pytest.mark.parametrize("k,n,opts", [(31, 4_300_000, {}), (63, 4_300_000, {}), (31, 2_500_000, {"fine_slots": 4096})])
def test_small_lds(k, n, opts):
    kmers = uc.medium_model(23, n + n // 16, k)[:n]
    limit = uc.lib().uc_ctx_set_lds_limit
    limit.argtypes, limit.restype = [C.c_void_p, C.c_uint32], C.c_int
    with uc.Compactor(**opts) as c:
        want = c.compact(kmers, k, 11)
    with uc.Compactor(**opts) as c:
        assert limit(c._ctx, 65535) == uc.UC_E_ARG and limit(c._ctx, 65536) == uc.UC_OK
        for rep in range(2):
            assert c.compact(kmers, k, 11) == want, rep
