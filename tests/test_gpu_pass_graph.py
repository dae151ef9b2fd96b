"""Contraction passes that rank their chains over the chip (more sampled
splitters, or more tiles, than one workgroup takes): captured once and replayed
while sizes and buffers repeat.  Every replay, with eager work on another
context in between, gives the eager context's bytes."""
import pytest

import oracle
import unitigcoarsening_amd as uc

pytestmark = pytest.mark.gpu


# (k, l, k-mers, sample_log2): 41 k slots make more splitters than one workgroup ranks at sample_log2 1; 9.44 M slots more
# tiles at any
@pytest.mark.parametrize("k,l,n,sample", [(31, 11, 120_000, 1), (63, 13, 60_000, 1), (31, 11, 9_600_000, 0)])
def test_replays_match_eager(k, l, n, sample):
    kmers, small = uc.medium_model(31, n, k), uc.medium_model(33, 3_000, 31)
    with uc.Compactor(sample_log2=sample, profile=True) as p:
        p.compact(kmers, k, l)
        assert "k_chain_round" in p.kernel_stats() and "k_chain_one" not in p.kernel_stats()
    with uc.Compactor(sample_log2=sample) as g, uc.Compactor(sample_log2=sample, eager=True) as e:
        want = e.compact(kmers, k, l)
        g.load(kmers, k)
        for rep in range(4):
            g.compact_loaded(l)
            assert g.text() == want, rep
            e.compact(small, 31, 11)
    if n < 1_000_000:
        text, _, _ = oracle.textbook(kmers, k)
        assert uc.sorted_lines(want) == uc.sorted_lines(text)
