"""lvl2 -> lvl1 key switching on the matrix cores (csrc/iks21.hip) against the
oracle (IdentityKeySwitch<lvl21param>, TFHEpp/src/keyswitch.cpp:12-48), word
for word: batch sizes around the workgroups' 128, 256 and 512 ciphertexts and
the splits of the digit positions, and mask words at the ends of the digits
and of their rounding.
"""

import numpy as np
import pytest

import cufhedb_amd as F

import _oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ksk21(full636):
    k, _ = full636
    # the context's KSK 21 was generated on the device from this seed; the
    # host generator gives the same key word for word
    return F.keygen_ksk(k.sk, 21, k.seed + 5)


def edge_words(rng, rows):
    """lvl2 words: row 0 zero, row 1 all ones, row 2 the largest word below a
    rounding step, row 3 one step, then every digit 7, every digit 4, uniform."""
    c = rng.integers(0, 1 << 64, (rows, F.LVL2_N + 1), dtype=np.uint64)
    for row, word in enumerate((0, (1 << 64) - 1, (1 << 33) - 1, 1 << 33,
                                0xfffffffc << 32, int("100" * 10, 2) << 34)):
        if row < rows:
            c[row] = word
    return c


@pytest.mark.parametrize("B", [1, 7, 128, 129, 256, 257, 512, 513, 1025])
def test_matches_oracle(full636, ksk21, B):
    _, ctx = full636
    rng = np.random.default_rng(B)
    c = edge_words(rng, B)
    out = ctx.iks(21, c)
    for b in sorted({0, 1, 2, 3, 4, 5, 6, 127, 128, 255, 256, 511, 512, B // 2, B - 1} & set(range(B))):
        assert np.array_equal(out[b], O.iks64(c[b], ksk21, F.LVL1_N, 10, 3)), (B, b)


def test_reloaded_key(full636, ksk21):
    """A key loaded from the host switches like the one generated on the
    device, and replaces the one before it."""
    k, ctx = full636
    c = edge_words(np.random.default_rng(9), 40)
    other = F.Context(k.params)
    try:
        other.load_ksk(21, np.zeros_like(ksk21))
        body = (c[:, F.LVL2_N] + np.uint64(1 << 31)) >> np.uint64(32)
        want = np.zeros((40, F.LVL1_N + 1), np.uint32)
        want[:, F.LVL1_N] = body.astype(np.uint32)
        assert np.array_equal(other.iks(21, c), want)
        other.load_ksk(21, ksk21)
        assert np.array_equal(other.iks(21, c), ctx.iks(21, c))
    finally:
        other.close()
