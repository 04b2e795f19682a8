"""Key switches 10 and 20 in the gather form (large batches, csrc/iks.hip)
against the whole-row form, word for word, and kind 10 against the oracle
(IdentityKeySwitch, TFHEpp/src/keyswitch.cpp:12-48): batches at the form's
first size and around its 4096 ciphertexts a workgroup, output widths around
its 16 columns, and mask words at the ends of the digits and their rounding.
"""

import numpy as np
import pytest

import cufhedb_amd as F

import _oracle as O

pytestmark = pytest.mark.gpu
KNOB = {10: F.TUNE_IKS_SPLIT, 20: F.TUNE_IKS20_SPLIT}


def words(rng, kind, rows):
    """Random TLWEs; the first rows all zero, all ones, just below and at a
    rounding step of the 20 digit bits, digits 1 and 1023."""
    w = 32 if kind == 10 else 64
    dt = np.uint32 if kind == 10 else np.uint64
    n = F.LVL1_N if kind == 10 else F.LVL2_N
    c = rng.integers(0, 1 << w, (rows, n + 1), dtype=np.uint64).astype(dt)
    step = 1 << (w - 21)
    for row, x in enumerate((0, (1 << w) - 1, step - 1, step, (1 << 10 | 1023) << (w - 20))):
        c[row] = dt(x)
    return c


def both(ctx, kind, c):
    """The default form and the whole-row form (four workgroups each)."""
    got = ctx.iks(kind, c)
    ctx.set_tune_table([(1, 4)], knob=KNOB[kind])
    try:
        return got, ctx.iks(kind, c)
    finally:
        ctx.set_tune_table([], knob=KNOB[kind])


@pytest.mark.parametrize("kind,B", [(10, 2400), (10, 4096), (10, 4097), (10, 8200), (20, 2048),
                                    (20, 4097)])
def test_gather_equals_rows(full672, kind, B):
    k, ctx = full672
    c = words(np.random.default_rng(B + kind), kind, B)
    got, want = both(ctx, kind, c)
    assert np.array_equal(got, want)
    if kind == 10:
        for b in {0, 1, 2, 3, 4, 5, 1023, 1024, 2399, B - 1}:
            assert np.array_equal(got[b], O.iks32(c[b], k.ksk10, k.n0)), b


@pytest.mark.parametrize("n0", [1, 15, 16, 31, 1024])
def test_gather_output_widths(n0):
    p = F.preset(F.PRESET_CFG636)
    p.n0 = n0
    p.key0_hw = min(p.key0_hw, n0)
    sk = F.SecretKeys(p, 51 + n0)
    ctx = F.Context(p)
    try:
        ctx.keygen_ksk(10, sk, 52 + n0)
        got, want = both(ctx, 10, words(np.random.default_rng(n0), 10, 2401))
        assert np.array_equal(got, want)
    finally:
        ctx.close()
