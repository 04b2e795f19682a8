"""Where key switches 10 and 20 turn to the gather form (csrc/iks.hip): around
the line at several output widths the default takes no longer than the
whole-row form, and both give the same words on either side of it.
"""

import ctypes

import numpy as np
import pytest

import cufhedb_amd as F

from test_gpu_iks_gather import KNOB, both, words

pytestmark = pytest.mark.gpu


def ms(ctx, kind, x, out, B, split):
    ctx.set_tune_table([(1, split)] if split else [], knob=KNOB[kind])
    best = []
    for _ in range(5):
        t = ctypes.c_float()
        F.check(F.lib().fhe_timer_start(ctx.h, None))
        for _ in range(4):
            F.check(F.lib().fhe_iks_dev(ctx.h, kind, x.ptr, out.ptr, B, None))
        F.check(F.lib().fhe_timer_stop(ctx.h, None, ctypes.byref(t)))
        best.append(t.value / 4)
    ctx.set_tune_table([], knob=KNOB[kind])
    return min(best)


@pytest.mark.parametrize("n0", [100, 255, 511, 636])
@pytest.mark.parametrize("kind", [10, 20])
def test_default_is_not_the_slower_form(n0, kind):
    """The whole-row form is timed with four workgroups a ciphertext, 2 to 4 %
    slower than its eight; a tenth more than that is the gather form taken too
    early (up to 1.3 times with one line for all widths)."""
    p = F.preset(F.PRESET_CFG636)
    p.n0 = n0
    p.key0_hw = min(p.key0_hw, n0)
    sk = F.SecretKeys(p, 61 + n0)
    ctx = F.Context(p)
    try:
        ctx.keygen_ksk(kind, sk, 62 + n0)
        c = words(np.random.default_rng(n0 + kind), kind, 2360)
        x, out = F.DeviceBuffer.from_array(c), F.DeviceBuffer(c.shape[0] * (n0 + 1) * 4)
        for B in (1699, 1700, 1850, 1990, 2100, 2260, 2349, 2350):
            a, b = (ms(ctx, kind, x, out, B, s) for s in (0, 4))
            assert a < 1.1 * b, (B, a, b)
        for B in (1950, 2290, 2350):
            got, want = both(ctx, kind, c[:B])
            assert np.array_equal(got, want), B
        x.free()
        out.free()
    finally:
        ctx.close()
