"""The two kernels behind two waves per polynomial (csrc/pbs_lvl1w2.hip): a
compute unit per ciphertext up to 512 of them, two waves per ciphertext beyond.
Both compute every value by the same operations, so a ciphertext's words do not
depend on the batch it is in, and a batch far beyond the line, which a table
tuned at small sizes only also sends here, takes the form that fills the GPU.
"""

import ctypes

import numpy as np
import pytest

import cufhedb_amd as F

from test_gpu_lvl1 import z8_testvector

pytestmark = pytest.mark.gpu
KNOB = F.TUNE_PBS1_WAVES


@pytest.fixture
def two_waves(ctx636):
    ctx636.set_tune_table([(1, 2)], knob=KNOB)
    yield ctx636
    ctx636.set_tune_table([], knob=KNOB)


def inputs(k, B, seed):
    rng = np.random.default_rng(seed)
    c0 = k.enc_lvl0((rng.integers(0, 8, B) << 28).astype(np.uint32), index0=91_000)
    c0[1] = 0                     # no step rotates
    c0[2, 1:] = 0                 # only the first
    c0[3, :-1] = 0xFFFFFFFF       # rounds to no rotation anywhere
    return c0, np.stack([z8_testvector(rng.integers(0, 8, 8)) for _ in range(B)])


def test_words_do_not_depend_on_the_batch(keys636, two_waves):
    c0, tvs = inputs(keys636, 513, 1)
    small = two_waves.pbs_lvl01(c0[:512], tvs[:512])
    large = two_waves.pbs_lvl01(c0, tvs)
    assert np.array_equal(large[:512], small)
    assert np.array_equal(two_waves.pbs_lvl01(c0[512:], tvs[512:])[0], large[512])
    # the accumulators too (no sample extraction, one table for all)
    acc = two_waves.blind_rotate_lvl01(c0, tvs[0])
    assert np.array_equal(two_waves.blind_rotate_lvl01(c0[:5], tvs[0]), acc[:5])


def test_large_batch_under_a_small_table(keys636, two_waves):
    """4096 ciphertexts with two waves each take about 1.2 times one wave's
    time (1.7 with a compute unit per ciphertext)."""
    ctx, B = two_waves, 4096
    c0 = keys636.enc_lvl0(np.zeros(B, np.uint32), index0=92_000)
    x, tv = F.DeviceBuffer.from_array(c0), F.DeviceBuffer.from_array(z8_testvector(np.arange(8)))
    out = F.DeviceBuffer(B * (F.LVL1_N + 1) * 4)

    def ms(waves):
        ctx.set_tune_table([(1, waves)], knob=KNOB)
        best = []
        for _ in range(4):
            t = ctypes.c_float()
            F.check(F.lib().fhe_timer_start(ctx.h, None))
            F.check(F.lib().fhe_pbs_lvl01_dev(ctx.h, x.ptr, tv.ptr, 0, out.ptr, B, None))
            F.check(F.lib().fhe_timer_stop(ctx.h, None, ctypes.byref(t)))
            best.append(t.value)
        return min(best)

    one, two = ms(1), ms(2)
    print(f"\n  4096 lvl1 bootstraps: one wave {one:.1f} ms, two {two:.1f} ms")
    assert two < 1.45 * one
    for b in (x, tv, out):
        b.free()
