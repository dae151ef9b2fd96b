"""k-mer lines with bytes other than A, C, G and T, in any place: the device
parser equals the host parser and the oracle's, and refuses what they refuse."""
import random

import numpy as np
import pytest

import oracle
import unitigcoarsening_amd as uc

pytestmark = pytest.mark.gpu

OTHER = [b for b in range(256) if b != ord("\n") and chr(b) not in "ACGT"]


def parse(text, k):
    with uc.Compactor() as c:
        c.load_text(text, k)
        return c.loaded(k)


@pytest.mark.parametrize("k", [2, 3, 4, 5, 15, 16, 17, 31, 32, 33, 47, 48, 63, 64])
def test_other_bytes(k):
    rng = random.Random(k)
    base = [bytes(rng.choice(b"ACGT") for _ in range(k)) for _ in range(2_000)]
    lines = []
    for i, s in enumerate(base):
        s = bytearray(s)
        for _ in range(rng.choice([0, 1, 1, 2, k])):
            s[rng.randrange(k)] = rng.choice(OTHER)
        if i < 2 * k:  # each place, '\r' among them
            s[i % k] = ord("\r") if i < k else ord("N")
        # (a '\r' as the last byte before a line end belongs to the line end)
        tail = bytes(rng.choice(b"ACGT \t\r0x") for _ in range(rng.choice([0, 0, 1, 5]))) + rng.choice([b"", b"", b"\r"])
        lines.append(bytes(s) + (tail or (b"" if s[-1] != 13 else b"7")))
    text = b"%d\n" % len(lines) + b"\n".join(lines) + b"\n"
    want = uc.parse_text(text, k)
    assert want.shape[0] == len(lines) and np.array_equal(want, oracle.parse_text(text, k))
    assert np.array_equal(parse(text, k), want)
    # the last line up to the text's last byte, and lines that are short by one: of letters, of others, by a '\r'
    assert np.array_equal(parse(text.rstrip(b"\r\n") + (b"" if len(lines[-1].rstrip(b"\r")) >= k else b"7"), k)[-1], want[-1])
    for short in (base[0][:-1], b"n" * (k - 1), base[0][:-1] + b"\r"):
        for bad in (text + short + b"\nACGT" + base[1] + b"\n", text + short):
            with pytest.raises(uc.UcError) as e:
                uc.parse_text(bad, k)
            assert e.value.status == uc.UC_E_FORMAT
            with pytest.raises(uc.UcError) as e:
                parse(bad, k)
            assert e.value.status == uc.UC_E_FORMAT
