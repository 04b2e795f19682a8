"""The calls whose time matters to a program that uses this library: single
operators, key switches, bootstraps and whole encrypted filters, from one
ciphertext to 2^14 rows.

A case is a plain dict.  ``prepare`` builds what a server program holds
before the call: a context with the keys that the call needs (one per
parameter set, kept for the life of the process, as a server keeps them) and
freshly encrypted inputs; ``run`` is one call through the public entry points
on the context's stream; ``work`` is what the call cannot do without.

Every output is a batch of ciphertexts: torus words, which are whole numbers
modulo 2^32 or 2^64 (viewed as signed integers of the same width), so two
builds are compared word for word and there is no floating output that an
``exact`` would describe.

Parameter sets: "ref672" (n0 = 672, the reference's set) and "cfg636"
(n0 = 636); both use lvl1 N = 1024, l = 3, Bgbit = 6 and lvl2 N = 2048,
l = 4, Bgbit = 9.  A bootstrap is n0 external products with their transforms.
"""

import math
from types import SimpleNamespace

import numpy as np
import torch

import cufhedb_amd as F
from cufhedb_amd import queries as Q

W1, W2 = F.LVL1_N + 1, F.LVL2_N + 1
PRESETS = {"ref672": F.PRESET_REF672, "cfg636": F.PRESET_CFG636}
N0 = {"ref672": 672, "cfg636": 636}
DIGIT_BITS = 4


def listed():
    return [
        # one gate through the host-array call: a program that evaluates a
        # circuit gate by gate waits for each one
        {"name": "gate_host_1", "op": "gate_host", "set": "ref672", "rows": 1, "gate": F.GATE_NAND},
        # one layer of a circuit over a column, operands resident on the device
        {"name": "gate_3000", "op": "gate", "set": "ref672", "rows": 3000, "gate": F.GATE_AND},
        # table lookups over a large batch, one table for all rows
        {"name": "pbs1_8192", "op": "pbs1", "set": "cfg636", "rows": 8192, "own_tables": False},
        # an odd, middling batch in which every row looks up its own table
        {"name": "pbs1_777_own", "op": "pbs1", "set": "ref672", "rows": 777, "own_tables": True},
        # lvl2 lookups: the few rows of an interactive query, and a column
        {"name": "pbs2_61", "op": "pbs2", "set": "ref672", "rows": 61, "own_tables": False},
        {"name": "pbs2_4096", "op": "pbs2", "set": "ref672", "rows": 4096, "own_tables": False},
        # the key switch in front of every lvl1 bootstrap, at a column's size
        {"name": "iks10_8192", "op": "iks", "set": "ref672", "rows": 8192, "kind": 10},
        # lvl2 -> lvl1 results of a small filter, and of a 2^14-row column
        {"name": "iks21_100", "op": "iks", "set": "ref672", "rows": 100, "kind": 21},
        {"name": "iks21_16384", "op": "iks", "set": "ref672", "rows": 16384, "kind": 21},
        # whole filters: TPC-H Q1's group predicates over a small table,
        {"name": "q1_256", "op": "q1", "set": "ref672", "rows": 256},
        # x <= t on 20-bit values with an encrypted threshold,
        {"name": "range20_300", "op": "range", "set": "ref672", "rows": 300, "bits": 20},
        # and x <= t on 20-bit values with a public threshold, digit by digit
        {"name": "digits20_1000", "op": "digits", "set": "cfg636", "rows": 1000, "digits": 5},
    ]


#: op -> (smallest, largest rows) of the ranges that the listed cases stand for
ROWS = {"gate_host": (1, 64), "gate": (1, 8192), "pbs1": (1, 8192), "pbs2": (1, 4096),
        "iks10": (1, 16384), "iks20": (1, 8192), "iks21": (1, 16384), "q1": (1, 512),
        "range": (1, 300), "digits": (1, 900)}


def draw(rng):
    op = rng.choice(["gate_host", "gate", "gate", "pbs1", "pbs1", "pbs2", "pbs2", "iks", "iks",
                     "iks", "q1", "range", "digits"])
    c = {"op": op, "set": rng.choice(sorted(PRESETS))}
    if op == "iks":
        c["kind"] = rng.choice([10, 20, 21])
    lo, hi = ROWS["iks%d" % c["kind"] if op == "iks" else op]
    c["rows"] = min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))
    if op in ("gate", "gate_host"):
        c["gate"] = rng.choice([F.GATE_NAND, F.GATE_AND, F.GATE_OR, F.GATE_NOR, F.GATE_XNOR])
    elif op in ("pbs1", "pbs2"):
        c["own_tables"] = rng.random() < 0.3
    elif op == "range":
        c["set"] = "ref672"  # the peeling chain's margins need the reference set
        c["bits"] = rng.choice([8, 12, 16, 20])
    elif op == "digits":
        c["digits"] = rng.randint(2, 5)
    elif op == "q1":
        c["set"] = "ref672"
    return c


# ------------------------------------------------------------------- keys
class Server:
    """A context with the keys loaded so far, and the secret keys its
    client encrypts under."""

    def __init__(self, name):
        self.params = F.preset(PRESETS[name])
        self.sk = F.SecretKeys(self.params, 20_001)
        self.ctx = F.Context(self.params)
        self.have = set()

    def need(self, *keys):
        for k in keys:
            if k in self.have:
                continue
            if k == "bk1":
                self.ctx.load_bk(1, F.keygen_bk_lvl01(self.sk, 20_002), F.BK_INT)
            elif k == "bk2":
                self.ctx.load_bk(2, F.keygen_bk_lvl02(self.sk, 20_003), F.BK_INT)
            else:
                self.ctx.keygen_ksk(k, self.sk, 20_004 + k)
            self.have.add(k)
        return self


_servers = {}


def server(name):
    if name not in _servers:
        _servers[name] = Server(name)
    return _servers[name]


KEYS = {"gate_host": ("bk1", 10), "gate": ("bk1", 10), "pbs1": ("bk1",), "pbs2": ("bk2",),
        "q1": ("bk1", 10), "range": ("bk1", "bk2", 10, 20, 21), "digits": ("bk2", 20, 21)}


# ----------------------------------------------------------------- inputs
def dev(a):
    """A host array on the GPU, its unsigned words viewed as signed ones."""
    a = np.ascontiguousarray(a)
    return torch.from_numpy(a.view(np.int32 if a.itemsize == 4 else np.int64)).cuda()


class Col:
    """A device tensor as the query functions take a buffer (``.ptr``)."""

    def __init__(self, t):
        self.t = t
        self.ptr = t.data_ptr()


def empty(rows, level):
    return torch.empty((rows, W1 if level == 1 else W2),
                       dtype=torch.int32 if level == 1 else torch.int64, device="cuda")


def enc0(s, seed, values, bits):
    m = (np.asarray(values, np.uint64) << np.uint64(32 - bits - 1)).astype(np.uint32)
    return F.tlwe_encrypt_u32(seed, 0, s.sk.s0, m, s.params.alpha0)


def enc1(s, seed, values, bits):
    m = (np.asarray(values, np.uint64) << np.uint64(32 - bits - 1)).astype(np.uint32)
    return F.tlwe_encrypt_u32(seed, 0, s.sk.s1, m, s.params.alpha1)


def enc2(s, seed, values, bits):
    m = np.asarray(values, np.uint64) << np.uint64(64 - bits - 1)
    return F.tlwe_encrypt_u64(seed, 0, s.sk.s2, m, s.params.alpha2)


def truth(s, seed, bits):
    """LOGIC booleans: +mu (true) or -mu (false) at lvl1."""
    m = np.where(np.asarray(bits) != 0, F.LVL1_MU, (1 << 32) - F.LVL1_MU).astype(np.uint32)
    return F.tlwe_encrypt_u32(seed, 0, s.sk.s1, m, s.params.alpha1)


def tables(rng, count, level):
    """Z_8 lookup tables as test vectors (one padding bit)."""
    n = F.LVL1_N if level == 1 else F.LVL2_N
    luts = rng.integers(0, 8, (count, 8))
    box = (np.arange(n) + n // 16) // (n // 8)
    v = np.where(box == 8, -luts[:, box % 8], luts[:, box % 8]).astype(np.int64)
    return (v << 28).astype(np.uint32) if level == 1 else (v << 60).astype(np.uint64)


def prepare(case, seed):
    op, rows = case["op"], case["rows"]
    s = server(case["set"]).need(*(KEYS[op] if op != "iks" else (case["kind"],)))
    rng = np.random.default_rng(seed)
    e = 1_000_003 * seed  # encryption randomness of this state's columns
    st = {"case": case, "ctx": s.ctx}
    if op in ("gate", "gate_host"):
        a, b = (truth(s, e + k, rng.integers(0, 2, rows)) for k in (1, 2))
        if op == "gate_host":
            st |= {"a": a, "b": b}
        else:
            st |= {"a": dev(a), "b": dev(b), "out": empty(rows, 1)}
    elif op in ("pbs1", "pbs2"):
        level = 1 if op == "pbs1" else 2
        tv = tables(rng, rows if case["own_tables"] else 1, level)
        st |= {"in": dev(enc0(s, e + 1, rng.integers(0, 8, rows), 3)), "tv": dev(tv),
               "stride": tv.shape[1] if case["own_tables"] else 0, "out": empty(rows, level)}
    elif op == "iks":
        kind, m = case["kind"], rng.integers(0, 16, rows)
        st |= {"in": dev(enc1(s, e + 1, m, 4) if kind == 10 else enc2(s, e + 1, m, 4)),
               "out": empty(rows, 1) if kind == 21 else
               torch.empty((rows, s.params.n0 + 1), dtype=torch.int32, device="cuda")}
    elif op == "q1":
        cols = ((rng.integers(0, 512, rows), 9), (rng.integers(0, 2, rows), 1),
                (rng.integers(0, 2, rows), 1), ([int(rng.integers(100, 400))], 9), ([1], 1))
        st["cols"] = [Col(dev(enc1(s, e + k, v, b))) for k, (v, b) in enumerate(cols)]
        # the filter's Q1Scratch on tensors, so that run can hand them out
        st["scratch"] = SimpleNamespace(rows=rows, p=[Col(empty(rows, 1)) for _ in range(5)],
                                        out=[Col(empty(rows, 1)) for _ in range(4)])
    elif op == "range":
        top = 1 << case["bits"]
        st |= {"x": Col(dev(enc2(s, e + 1, rng.integers(0, top, rows), case["bits"]))),
               "t": Col(dev(enc2(s, e + 2, [int(rng.integers(0, top))], case["bits"]))),
               "out": Col(empty(rows, 1))}
    else:
        n = case["digits"]
        top = 1 << (n * DIGIT_BITS)
        x = F.encrypt_digits(e + 1, 0, s.sk.s2, rng.integers(0, top, rows), n, DIGIT_BITS,
                             s.params.alpha2)
        st |= {"x": dev(x), "threshold": int(rng.integers(0, top)), "out": empty(rows, 1)}
    return st


# ------------------------------------------------------------------- call
def run(st):
    case, ctx, L = st["case"], st["ctx"], F.lib()
    op, rows = case["op"], case["rows"]
    if op == "gate_host":
        return ctx.gate(case["gate"], st["a"], st["b"]).view(np.int32)
    if op == "q1":
        ship, flag, status, date, one = st["cols"]
        s = Q.tpch_q1_filter(ctx, ship, flag, status, date, one, rows, scratch=st["scratch"])
        return [b.t for b in s.out]
    if op == "range":
        return Q.range_filter(ctx, st["x"], st["t"], rows, case["bits"], out_dev=st["out"]).t
    out = st["out"]
    if op == "gate":
        rc = L.fhe_gate_lvl1_dev(ctx.h, case["gate"], st["a"].data_ptr(), st["b"].data_ptr(),
                                 out.data_ptr(), F.LOGIC, rows, None)
    elif op == "pbs1":
        rc = L.fhe_pbs_lvl01_dev(ctx.h, st["in"].data_ptr(), st["tv"].data_ptr(), st["stride"],
                                 out.data_ptr(), rows, None)
    elif op == "pbs2":
        rc = L.fhe_pbs_lvl02_dev(ctx.h, st["in"].data_ptr(), st["tv"].data_ptr(), st["stride"],
                                 out.data_ptr(), rows, None)
    elif op == "iks":
        rc = L.fhe_iks_dev(ctx.h, case["kind"], st["in"].data_ptr(), out.data_ptr(), rows, None)
    else:
        rc = L.fhe_compare_digits_dev(ctx.h, F.CMP_LE, st["x"].data_ptr(), case["digits"],
                                      DIGIT_BITS, st["threshold"], 1, out.data_ptr(), F.LOGIC,
                                      rows, None)
    F.check(rc)
    return out


# ------------------------------------------------------------------- work
def bootstrap(n0, level):
    """(flops of one bootstrap, bytes of its key): per external product the
    row and column transforms at 5 M log2 M and the products at 8 M a pair."""
    m, rows = (512, 6) if level == 1 else (1024, 8)
    flops = n0 * ((rows + 2) * 5 * m * int(math.log2(m)) + rows * 2 * 8 * m)
    return flops, n0 * rows * 2 * m * 16


def switch_key(n0, kind, rows):
    """Bytes of the key rows that `rows` ciphertexts select: each distinct
    row once (uniform digits)."""
    positions, cand = (2048, 1023) if kind == 10 else (4096, 1023) if kind == 20 else (20480, 7)
    width = W1 if kind == 21 else n0 + 1
    return positions * cand * -math.expm1(rows * math.log1p(-1 / (cand + 1))) * width * 4


def work(case):
    n0, op, r = N0[case["set"]], case["op"], case["rows"]
    lv0, lv1, lv2 = 4 * (n0 + 1), 4 * W1, 8 * W2
    f1, k1 = bootstrap(n0, 1)
    f2, k2 = bootstrap(n0, 2)
    if op in ("gate", "gate_host"):
        return {"bytes": 3 * r * lv1 + k1 + switch_key(n0, 10, r), "flops": r * f1}
    if op == "pbs1":
        return {"bytes": r * (lv0 + lv1) + (r if case["own_tables"] else 1) * 4096 + k1,
                "flops": r * f1}
    if op == "pbs2":
        return {"bytes": r * (lv0 + lv2) + (r if case["own_tables"] else 1) * 16384 + k2,
                "flops": r * f2}
    if op == "iks":
        kind = case["kind"]
        return {"bytes": r * ((lv1 if kind == 10 else lv2) + (lv1 if kind == 21 else lv0)) +
                switch_key(n0, kind, r), "flops": 0.0}
    if op == "q1":
        # the date's comparison (a chain of five), the two flags', six ANDs
        return {"bytes": 7 * r * lv1 + k1 + switch_key(n0, 10, 13 * r), "flops": 13 * r * f1}
    if op == "range":
        # one sign bit more, peeled five bits a time down to nine (two lvl2
        # bootstraps each), then at most three lvl1 bootstraps
        peels = max(0, -(-(case["bits"] + 1 - 9) // 5))
        return {"bytes": r * (lv2 + lv1) + k1 + (k2 if peels else 0) +
                switch_key(n0, 20, 2 * peels * r) + switch_key(n0, 21, r) +
                switch_key(n0, 10, 3 * r), "flops": r * (2 * peels * f2 + 3 * f1)}
    n = case["digits"]
    return {"bytes": r * (n * lv2 + lv1) + k2 + switch_key(n0, 20, (n + 1) * r) +
            switch_key(n0, 21, r), "flops": r * (n + 1) * f2}
