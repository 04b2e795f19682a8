"""Small-batch bootstraps at the edges of their step list: lvl0 dimensions
around a wave (64) and at the limit (1024), mask words that round to a
rotation of zero (skipped CMUX steps) in some, all and none of the positions;
and the lvl2 small-batch kernel (up to 256 ciphertexts) against the large one.

Bars: with no rotation at all the output is the rotated test vector itself,
word for word; otherwise the phase is within 2^26 (lvl1) or 2^40 (lvl2) of
the oracle's (TFHEpp gatebootstrapping.hpp:15-43), the bars of every bootstrap
here.  The two lvl2 kernels agree word for word.
"""

import numpy as np
import pytest

import cufhedb_amd as F

import _oracle as O
from test_gpu_lvl1 import z8_testvector

pytestmark = pytest.mark.gpu


def params_with(n0):
    p = F.preset(F.PRESET_CFG636)
    p.n0 = n0
    p.key0_hw = min(p.key0_hw, n0)
    return p


def masks(rng, n0, rows, nbit):
    """Uniform lvl0 words; row 0 all zero rotations (mask words below half a
    step of the switch to 2N = 2^(nbit + 1)), row 1 alternating, row 2 only the
    last step, the rest none."""
    c = rng.integers(0, 1 << 32, (rows, n0 + 1), dtype=np.uint64).astype(np.uint32)
    small = rng.integers(0, 1 << (30 - nbit), (rows, n0 + 1), dtype=np.uint64).astype(np.uint32)
    c[0, :n0] = small[0, :n0]
    c[1, :n0:2] = small[1, :n0:2]
    c[2, : n0 - 1] = small[2, : n0 - 1]
    return c


@pytest.mark.parametrize("n0", [1, 63, 64, 65, 1024])
def test_lvl1_step_list_edges(n0):
    p = params_with(n0)
    sk = F.SecretKeys(p, 31 + n0)
    bk = F.keygen_bk_lvl01(sk, 32 + n0)
    ctx = F.Context(p)
    try:
        ctx.load_bk(1, bk, F.BK_INT)
        rng = np.random.default_rng(n0)
        c = masks(rng, n0, 5, 10)
        tv = z8_testvector(rng.integers(0, 8, 8))
        out = ctx.pbs_lvl01(c, tv)
        bkfft = O.bk_to_fft32(bk)
        for b in range(5):
            want = O.pbs32(c[b], bkfft, tv)
            if b == 0:
                assert np.array_equal(out[b], want)
            gap = O.tdiff32(F.tlwe_phase_u32(out[b], sk.s1), F.tlwe_phase_u32(want, sk.s1))
            assert abs(int(gap[0])) < 1 << 26, (n0, b)
    finally:
        ctx.close()


def lvl2_testvector(rng):
    n = F.LVL2_N
    lut = rng.integers(0, 8, 8)
    box = (np.arange(n) + n // 16) // (n // 8)
    return (np.where(box == 8, -lut[box % 8], lut[box % 8]).astype(np.int64) << 60).astype(np.uint64)


@pytest.mark.parametrize("n0", [1, 65, 1024])
def test_lvl2_step_list_edges(n0):
    p = params_with(n0)
    sk = F.SecretKeys(p, 41 + n0)
    bk = F.keygen_bk_lvl02(sk, 42 + n0)
    ctx = F.Context(p)
    try:
        ctx.load_bk(2, bk, F.BK_INT)
        rng = np.random.default_rng(n0)
        c = masks(rng, n0, 5, 11)
        tv = lvl2_testvector(rng)
        out = ctx.pbs_lvl02(c, tv)
        bkfft = O.bk_to_fft64(bk)
        for b in range(5):
            want = O.pbs64(c[b], bkfft, tv)
            if b == 0:
                assert np.array_equal(out[b], want)
            gap = O.tdiff64(O.tlwe_phase64(out[b], sk.s2), O.tlwe_phase64(want, sk.s2))
            assert abs(int(np.ravel(gap)[0])) < 1 << 40, (n0, b)
    finally:
        ctx.close()


def test_lvl2_small_and_large_kernels_agree(full636, rng):
    k, ctx = full636
    c = k.enc_lvl0((rng.integers(0, 8, 257) << 28).astype(np.uint32), index0=90000)
    tvs = np.stack([lvl2_testvector(rng) for _ in range(257)])
    for tv in (tvs[0], tvs):
        large = ctx.pbs_lvl02(c, tv)
        small = ctx.pbs_lvl02(c[:256], tv if tv.ndim == 1 else tv[:256])
        assert np.array_equal(large[:256], small)
    acc = ctx.blind_rotate_lvl02(c[:3], tvs[0])
    assert np.array_equal(acc, ctx.blind_rotate_lvl02(c, tvs[0])[:3])
