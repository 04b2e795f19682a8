"""Small bootstraps next to a long launch on another stream of the same context:
they get in between its workgroups instead of waiting for its end, and give the
words that they give alone.
"""

import numpy as np
import pytest
import torch

import cufhedb_amd as F

from test_gpu_lvl1 import z8_testvector

pytestmark = pytest.mark.gpu


class Calls:
    """Bootstraps of the first rows of one batch on a given torch stream."""

    def __init__(self, k, ctx):
        rng = np.random.default_rng(5)
        m = (rng.integers(0, 8, 16384) << 28).astype(np.uint32)
        self.ctx = ctx
        self.x = torch.from_numpy(k.enc_lvl0(m, index0=95_000).view(np.int32)).cuda()
        self.tv = {1: torch.from_numpy(z8_testvector(rng.integers(0, 8, 8)).view(np.int32)).cuda(),
                   2: torch.from_numpy(rng.integers(-1 << 63, 1 << 63, F.LVL2_N)).cuda()}

    def out(self, level, B):
        return torch.zeros((B, (F.LVL1_N if level == 1 else F.LVL2_N) + 1),
                           dtype=torch.int32 if level == 1 else torch.int64, device="cuda")

    def go(self, level, B, out, stream):
        f = F.lib().fhe_pbs_lvl01_dev if level == 1 else F.lib().fhe_pbs_lvl02_dev
        F.check(f(self.ctx.h, self.x.data_ptr(), self.tv[level].data_ptr(), 0, out.data_ptr(), B,
                  stream.cuda_stream))


@pytest.fixture(scope="module")
def calls(full672):
    return Calls(*full672)


@pytest.mark.parametrize("big,nb,small,ns", [(2, 4096, 1, 1), (2, 4096, 1, 511), (2, 4096, 2, 1),
                                             (2, 4096, 2, 256), (1, 16384, 1, 1), (1, 16384, 1, 32)])
def test_small_call_does_not_wait_for_the_long_one(calls, big, nb, small, ns):
    c = calls
    s1 = torch.cuda.Stream()
    alone, lone = c.out(small, ns), c.out(big, nb)
    c.go(small, ns, alone, s1)
    best = []
    # streams share a few hardware queues: one of these is not in s1's
    for s2 in [torch.cuda.Stream() for _ in range(4)]:
        beside = c.out(small, ns)
        e = [torch.cuda.Event(enable_timing=True) for _ in range(3)]
        torch.cuda.synchronize()
        e[0].record(s1)
        c.go(big, nb, lone, s1)
        e[1].record(s1)
        c.go(small, ns, beside, s2)
        e[2].record(s2)
        torch.cuda.synchronize()
        best.append((e[0].elapsed_time(e[2]), e[0].elapsed_time(e[1])))
        assert torch.equal(alone, beside)
    small_ms, long_ms = min(best)
    print(f"\n  long {long_ms:.1f} ms, small {small_ms:.1f} ms")
    assert small_ms < 0.8 * long_ms
    # the long launch's own words, with and without company
    again = c.out(big, nb)
    c.go(big, nb, again, s1)
    torch.cuda.synchronize()
    assert torch.equal(lone, again)


def test_beside_an_open_capture(calls):
    """Neither the long launch nor the small one touches a capture that another
    stream has open, and a small call recorded into one replays as it runs."""
    c = calls
    s1, s2, s3 = (torch.cuda.Stream() for _ in range(3))
    alone, beside, rec, lone = c.out(2, 3), c.out(2, 3), c.out(2, 3), c.out(2, 1000)
    c.go(2, 3, alone, s2)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s3):
        c.go(2, 1000, lone, s1)
        c.go(2, 3, beside, s2)
        c.go(2, 1000, lone, s3)  # recorded, so not in flight
        c.go(2, 3, rec, s3)
    torch.cuda.synchronize()
    assert torch.equal(alone, beside)
    for _ in range(3):
        rec.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(alone, rec)
