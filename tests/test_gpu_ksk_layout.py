"""Key switches 10 and 20 from device rows at whole 128-byte lines
(csrc/iks.hip): output widths around the lines' 32 words, batches on both sides
of the gather form's first size, and few enough ciphertexts to be split over
more workgroups each, against the oracle (IdentityKeySwitch,
TFHEpp/src/keyswitch.cpp:12-48), word for word.  The keys are random words, so
a row read from the wrong place shows.
"""

import numpy as np
import pytest

import cufhedb_amd as F

import _oracle as O

pytestmark = pytest.mark.gpu


def context(n0):
    p = F.preset(F.PRESET_CFG636)
    p.n0 = n0
    p.key0_hw = min(p.key0_hw, n0)
    return F.Context(p)


@pytest.mark.parametrize("n0", [30, 31, 32, 95])
def test_row_lines_kind10(n0):
    rng = np.random.default_rng(n0)
    ksk = rng.integers(0, 1 << 32, 1024 * 2 * 1023 * (n0 + 1), np.uint32)
    ctx = context(n0)
    try:
        ctx.load_ksk(10, ksk)
        for B in (3, 1999, 2000):
            c = rng.integers(0, 1 << 32, (B, F.LVL1_N + 1), np.uint32)
            c[0] = 0xFFFFFFFF
            c[-1] = 1 << 11
            got = ctx.iks(10, c)
            for b in {0, 1, B // 2, B - 1}:
                assert np.array_equal(got[b], O.iks32(c[b], ksk, n0)), (B, b)
    finally:
        ctx.close()


def test_first_gather_size_kind20():
    n0 = 33
    rng = np.random.default_rng(20)
    ksk = rng.integers(0, 1 << 32, 2048 * 2 * 1023 * (n0 + 1), np.uint32)
    ctx = context(n0)
    try:
        ctx.load_ksk(20, ksk)
        c = rng.integers(0, 1 << 64, (1701, F.LVL2_N + 1), np.uint64)
        c[0] = (1 << 64) - 1
        c[1699] = 1 << 43
        want = {b: O.iks64(c[b], ksk, n0, 2, 10) for b in (0, 1, 850, 1698, 1699, 1700)}
        for B in (1699, 1700, 1701):
            got = ctx.iks(20, c[:B])
            for b, w in want.items():
                assert b >= B or np.array_equal(got[b], w), (B, b)
    finally:
        ctx.close()


@pytest.mark.parametrize("kind", [10, 20])
def test_few_ciphertexts(kind):
    """64, 32, 16 and 8 workgroups a ciphertext."""
    n0, wide = 40, kind == 20
    n = F.LVL2_N if wide else F.LVL1_N
    rng = np.random.default_rng(kind + 1)
    ksk = rng.integers(0, 1 << 32, n * 2 * 1023 * (n0 + 1), np.uint32)
    ctx = context(n0)
    try:
        ctx.load_ksk(kind, ksk)
        c = rng.integers(0, 1 << (64 if wide else 32), (65, n + 1), np.uint64 if wide else np.uint32)
        c[0] = 0
        for B in (1, 2, 8, 9, 16, 17, 32, 33, 65):
            got = ctx.iks(kind, c[:B])
            for b in {0, B // 2, B - 1}:
                want = O.iks64(c[b], ksk, n0, 2, 10) if wide else O.iks32(c[b], ksk, n0)
                assert np.array_equal(got[b], want), (B, b)
    finally:
        ctx.close()
