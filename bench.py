"""Headline benchmark: batched lvl1 programmable bootstrapping on one MI355X.

Workload (one "step"): a batch of B = 8192 lvl0 LWE ciphertexts (n0 = 636,
uniform binary key, alpha0 = 2^-15) holding Z_8 plaintexts with one padding
bit, bootstrapped to lvl1 (N = 1024, k = 1, l = 3, Bgbit = 6) through a
random 8-entry lookup table: one fhe_pbs_lvl01_dev launch = BlindRotate +
SampleExtract for all B ciphertexts (TFHEpp GateBootstrappingTLWE2TLWEFFT).
Inputs, key and outputs stay resident in HBM during the timed region; the
time is taken with HIP events on the stream the kernel runs on.

Prints one JSON line (see the repository's measurement contract): PBS/s,
the roofline fraction of the dominant kernel, and a CPU baseline timed on
this host's cores.
"""

import argparse
import concurrent.futures as cf
import ctypes
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "lvl1 PBS/sec @batch 8192 (MFMA-split vs FP64); ms per 2^14-row encrypted query"
PEAK_FP64_TFLOPS = 78.6  # MI355X dense FP64 (vector and matrix)
N, L, BGBIT = 1024, 3, 6


def flops_per_pbs(n0):
    """FFT-based algorithmic flops of one lvl1 PBS (k = 1):
    n0 * [((k+1)l + (k+1)) * 5 (N/2) log2(N/2) + (k+1)l (k+1) * 8 (N/2)]."""
    M = N // 2
    return n0 * ((2 * L + 2) * 5 * M * 9 + 2 * L * 2 * 8 * M)


def z8_testvector(lut):
    j = np.arange(N)
    box = (j + 64) >> 7
    vals = np.array(lut, np.int64)[box % 8] << 28
    vals = np.where(box == 8, -vals, vals)
    return (vals % (1 << 32)).astype(np.uint32)


def load_traffic(variant, preset, batch):
    """HBM bytes per launch measured with rocprofv3 --pmc (committed summary)."""
    path = os.path.join(ROOT, "profiles", f"pbs_lvl01_{variant}_{preset}_b{batch}.traffic.json")
    if not os.path.exists(path):
        return None
    with open(path) as f:
        return json.load(f).get("hbm_bytes_per_launch")


def cpu_baseline(threads, seconds_budget=12.0):
    """Reference TFHEpp (oracle/_ref, compiled from the reference sources) PBS
    throughput on this host, falling back to the oracle's C restatement."""
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import _oracle as O
    import cufhedb_amd as F

    ref = O.ref()
    if ref is not None:
        p = F.preset(F.PRESET_REF672)
        kind, fn_name = "reference", "ref_pbs_lvl01"
    else:
        p = F.preset(F.PRESET_CFG636)
        kind, fn_name = "port", "orc_pbs_u32"
    sk = F.SecretKeys(p, 99)
    bkfft = O.bk_to_fft32(F.keygen_bk_lvl01(sk, 98))
    rng = np.random.default_rng(5)
    tv = z8_testvector(rng.integers(0, 8, 8))
    nsamp = 4 * threads
    c0 = F.tlwe_encrypt_u32(97, 0, sk.s0, (rng.integers(0, 8, nsamp) << 28).astype(np.uint32),
                            p.alpha0)
    n0 = p.n0

    def one(i):
        out = np.zeros(N + 1, np.uint32)
        row = np.ascontiguousarray(c0[i % nsamp])
        if kind == "reference":
            ref.ref_pbs_lvl01(O.P(out), O.P(row), O.P(bkfft), O.P(tv))
        else:
            O.orc().orc_pbs_u32(O.P(out), O.P(row), n0, O.P(bkfft), O.P(tv), N, 10, L, BGBIT)
        return 1

    # calibrate on one PBS, then size the sample to ~seconds_budget of CPU work
    t = time.perf_counter()
    one(0)
    per = time.perf_counter() - t
    total = max(threads, int(seconds_budget / max(per, 1e-4)))
    total = (total + threads - 1) // threads * threads
    with cf.ThreadPoolExecutor(threads) as ex:
        t = time.perf_counter()
        done = sum(ex.map(one, range(total)))
        wall = time.perf_counter() - t
    # one host thread over ~2 s of the same work (the per-core rate)
    n1 = max(4, int(2.0 / max(per, 1e-4)))
    t = time.perf_counter()
    for i in range(n1):
        one(i)
    wall1 = time.perf_counter() - t
    impl = ("TFHEpp GateBootstrappingTLWE2TLWEFFT<lvl01param> (spqlios FP64 FFT) compiled from "
            "the reference sources, its fixed n0=672" if kind == "reference" else
            "oracle C restatement, n0=636")
    return {
        "value": done / wall,
        "unit": "PBS/s",
        "cores": threads,
        "kind": kind,
        "sample": f"{done} lvl1 PBS ({impl}), one ciphertext per thread at a time, "
                  f"{wall:.2f} s wall on {threads} host threads",
        "single_thread": {"value": n1 / wall1, "unit": "PBS/s",
                          "sample": f"{n1} lvl1 PBS on one host thread in {wall1:.2f} s"},
    }


def gate_and_iks_rates(F, ctx, sk, p, B, reps, threads, seconds_budget=4.0):
    """The config-1 gate (HomNAND = lvl1 -> lvl0 key switch + PBS) and the
    lvl1 -> lvl0 key switch alone, at n0 = 672: the device path at batch B
    (HIP events) beside the compiled reference TFHEpp on `threads` host
    threads over a bounded sample (HomNAND<lvl1param>, IdentityKeySwitch
    <lvl10param>; gate.cpp:50-65, keyswitch.cpp:12-48), keys identical on both
    sides (the device key switch key regenerated into a buffer from the
    context's seed and copied to the host).  None when the compiled reference
    is not built."""
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import _oracle as O

    ref = O.ref()
    if ref is None:
        return None
    L_ = F.lib()
    rng = np.random.default_rng(29)
    mu, minus_mu = np.uint32(1 << 29), np.uint32((1 << 32) - (1 << 29))
    bits_a, bits_b = rng.integers(0, 2, B), rng.integers(0, 2, B)
    enc = lambda seed, bits: F.tlwe_encrypt_u32(
        seed, 0, sk.s1, np.where(bits == 1, mu, minus_mu).astype(np.uint32), 2.0 ** -25)
    ca, cb = enc(41, bits_a), enc(42, bits_b)
    da, db = F.DeviceBuffer.from_array(ca), F.DeviceBuffer.from_array(cb)
    dout = F.DeviceBuffer(B * (N + 1) * 4)
    d0 = F.DeviceBuffer(B * (p.n0 + 1) * 4)
    gate_ms = timed_on(F, ctx, lambda: F.check(L_.fhe_gate_lvl1_dev(
        ctx.h, F.GATE_NAND, da.ptr, db.ptr, dout.ptr, F.LOGIC, B, None)), reps)
    ph = F.tlwe_phase_u32(dout.to_array(np.uint32, (B, N + 1)), sk.s1).view(np.int32)
    gate_err = int(np.sum((ph > 0) != ((bits_a & bits_b) == 0)))
    iks_ms = timed_on(F, ctx, lambda: F.check(L_.fhe_iks_dev(ctx.h, 10, da.ptr, d0.ptr, B, None)),
                      reps)
    # the same key switching key on the host (5.6 GB)
    kbytes = N * 2 * 1023 * (p.n0 + 1) * 4
    dk = F.DeviceBuffer(kbytes + 256)
    ctx.keygen_ksk(10, sk, 20261206, out_dev=dk)
    ctx.sync()
    ksk = dk.to_array(np.uint32, ((kbytes + 256) // 4,))
    for b in (da, db, dout, d0, dk):
        b.free()
    bkfft = O.bk_to_fft32(F.keygen_bk_lvl01(sk, 20261213))
    n0 = p.n0

    def cpu_rate(fn):
        fn(0)
        t = time.perf_counter()
        fn(1)
        per = time.perf_counter() - t
        total = max(threads, int(seconds_budget / max(per, 1e-5)))
        total = (total + threads - 1) // threads * threads
        with cf.ThreadPoolExecutor(threads) as ex:
            t = time.perf_counter()
            done = sum(ex.map(fn, range(total)))
            wall = time.perf_counter() - t
        return done / wall, done, wall

    def nand(i):
        out = np.zeros(N + 1, np.uint32)
        ref.ref_hom_nand_lvl1(O.P(out), O.P(np.ascontiguousarray(ca[i % B])),
                              O.P(np.ascontiguousarray(cb[i % B])), O.P(bkfft), O.P(ksk))
        return 1

    def iks(i):
        out = np.zeros(n0 + 1, np.uint32)
        ref.ref_iks_lvl10(O.P(out), O.P(np.ascontiguousarray(ca[i % B])), O.P(ksk))
        return 1

    nand_rate, nand_n, nand_wall = cpu_rate(nand)
    iks_rate, iks_n, iks_wall = cpu_rate(iks)
    del ksk
    out = {
        "hom_nand": {"unit": "gates/s", "gpu": B / gate_ms * 1e3, "gpu_batch": B,
                     "gpu_errors": gate_err, "cpu": nand_rate,
                     "cpu_sample": f"{nand_n} HomNAND<lvl1param> in {nand_wall:.2f} s"},
        "iks_lvl10": {"unit": "key switches/s", "gpu": B / iks_ms * 1e3, "gpu_batch": B,
                      "cpu": iks_rate,
                      "cpu_sample": f"{iks_n} IdentityKeySwitch<lvl10param> in {iks_wall:.2f} s"},
        "cores": threads, "n0": int(n0),
    }
    print(f"bench: HomNAND n0={n0}: GPU {out['hom_nand']['gpu']:.0f} gates/s at batch {B} "
          f"({gate_err} errors), CPU {nand_rate:.0f} gates/s on {threads} threads; lvl1 -> lvl0 "
          f"key switch: GPU {out['iks_lvl10']['gpu']:.0f}/s, CPU {iks_rate:.0f}/s",
          file=sys.stderr, flush=True)
    return out


def operator_context(F, which=None):
    """A context with every key the operator layer uses, by default on the
    reference's own parameter set (n0 = 672, alpha0 = 2^-16).  The lvl2
    comparison chains need it: with n0 = 636 / alpha0 = 2^-15 the
    key-switched lvl0 noise sits about 3 sigma from the 6-bit windows'
    decision boundaries (the digit-wise comparison keeps 2^-6 of margin and
    also runs at n0 = 636)."""
    p = F.preset(F.PRESET_REF672 if which is None else which)
    sk = F.SecretKeys(p, 20261212)
    ctx = F.Context(p, 0)
    ctx.load_bk(1, F.keygen_bk_lvl01(sk, 20261213), F.BK_INT)
    ctx.load_bk(2, F.keygen_bk_lvl02(sk, 20261205), F.BK_INT)
    for kind, seed in ((10, 20261206), (20, 20261207), (21, 20261208)):
        ctx.keygen_ksk(kind, sk, seed)  # on the device; same key as keygen_ksk
    return ctx, sk, p


TUNE = {
    "iks21_tile": ("tile of the lvl2 -> lvl1 key switch (8, 16: 128 ciphertexts a workgroup, "
                   "32: 256, 64: 512)",
                   (32, 128, 512, 1024, 2048, 4096, 16384)),
    "pbs1_waves": ("waves per polynomial of the lvl1 blind rotation",
                   (64, 256, 512, 1024, 2048)),
    "iks_split": ("workgroups per ciphertext of the lvl1 -> lvl0 key switch",
                  (16, 64, 256, 1024, 4096, 16384)),
    "iks20_split": ("workgroups per ciphertext of the lvl2 -> lvl0 key switch",
                    (16, 64, 256, 1024, 4096, 16384)),
}
KNOBS = (("iks21_tile", "TUNE_IKS21_TILE"), ("pbs1_waves", "TUNE_PBS1_WAVES"),
         ("iks_split", "TUNE_IKS_SPLIT"), ("iks20_split", "TUNE_IKS20_SPLIT"))


def autotune(F, ctx):
    """Shapes measured on this GPU per batch size and kept in the context for
    the query pipelines: the lvl2 -> lvl1 key switch's tile, the lvl1 blind
    rotation's waves per polynomial and the lvl1 -> lvl0 and lvl2 -> lvl0
    key switches' workgroups per ciphertext (each tuned on its own key)."""
    out = {}
    for name, attr in KNOBS:
        knob = getattr(F, attr)
        what, batches = TUNE[name]
        res = ctx.autotune(batches, knob=knob)
        print(f"bench: autotuned {what}: {ctx.tune_table(knob=knob)}", file=sys.stderr,
              flush=True)
        out[name] = {"knob": what, "table": {str(b): t for b, (t, _) in res.items()},
                     "ms": {str(b): ms for b, (_, ms) in res.items()}}
    return out


def apply_tuning(F, ctx, tuned):
    for name, attr in KNOBS:
        knob = getattr(F, attr)
        ctx.set_tune_table(sorted((int(b), t) for b, t in tuned[name]["table"].items()),
                           knob=knob)


def timed_on(F, ctx, fn, reps):
    """Mean milliseconds of fn over `reps` runs after one untimed run (which
    also sizes the operator scratch), HIP events on the context stream."""
    L_ = F.lib()
    fn()
    ctx.sync()
    F.check(L_.fhe_timer_start(ctx.h, None))
    for _ in range(reps):
        fn()
    ms = ctypes.c_float()
    F.check(L_.fhe_timer_stop(ctx.h, None, ctypes.byref(ms)))
    return float(ms.value) / reps


def pbs_lvl01_rate(F, ctx, sk, p, B, reps):
    """FP64 lvl1 PBS/s at batch B on ctx's parameter set (the Z_8 workload
    of the headline), for the like-for-like line beside the CPU baseline,
    which runs the reference's own parameter set (n0 = 672)."""
    rng = np.random.default_rng(23)
    m = rng.integers(0, 8, B)
    lut = rng.integers(0, 8, 8)
    c0 = F.tlwe_encrypt_u32(31, 0, sk.s0, (m << 28).astype(np.uint32), p.alpha0)
    d_in, d_tv = F.DeviceBuffer.from_array(c0), F.DeviceBuffer.from_array(z8_testvector(lut))
    d_out = F.DeviceBuffer(B * (N + 1) * 4)
    L_ = F.lib()
    ms = timed_on(F, ctx, lambda: F.check(L_.fhe_pbs_lvl01_dev(ctx.h, d_in.ptr, d_tv.ptr, 0,
                                                                d_out.ptr, B, None)), reps)
    ph = F.tlwe_phase_u32(d_out.to_array(np.uint32, (B, N + 1)), sk.s1).view(np.int32)
    fails = int(np.sum(np.round(ph.astype(np.int64) / (1 << 28)).astype(np.int64) % 16 != lut[m]))
    for b in (d_in, d_tv, d_out):
        b.free()
    print(f"bench: fp64 lvl1 PBS at n0={p.n0}, batch {B}: {ms:.2f} ms, {B / ms * 1e3:.0f} PBS/s, "
          f"{fails} decryption failures", file=sys.stderr, flush=True)
    return {"workload": f"lvl1 PBS, batch {B}, n0={p.n0}, fp64 (same kernel as the headline)",
            "ms_per_step": ms, "pbs_per_s": B / ms * 1e3, "decrypt_failures": fails}


def run_compare_digits(F, ctx, sk, p, rows, reps):
    """x <= t for `rows` seeded uniform 20-bit values against a seeded public
    threshold, digit-wise: five 4-bit lvl2 digits per value, one lvl2 PBS per
    digit plus one combining PBS, lvl1 results (IKS lvl21)."""
    rng = np.random.default_rng(19)
    x = rng.integers(0, 1 << 20, rows).astype(np.uint64)
    t = int(rng.integers(0, 1 << 20))
    dx = F.DeviceBuffer.from_array(F.encrypt_digits(321, 0, sk.s2, x, 5, 4, p.alpha2))
    out = F.DeviceBuffer(rows * (N + 1) * 4)
    L_ = F.lib()
    ms = timed_on(F, ctx, lambda: F.check(L_.fhe_compare_digits_dev(
        ctx.h, F.CMP_LE, dx.ptr, 5, 4, t, 1, out.ptr, F.LOGIC, rows, None)), reps)
    ph = F.tlwe_phase_u32(out.to_array(np.uint32, (rows, N + 1)), sk.s1).view(np.int32)
    errors = int(np.sum((ph > 0) != (x <= t)))
    dx.free()
    out.free()
    print(f"bench: digit-wise compare {rows} rows, n0={p.n0}: {ms:.1f} ms/query, {errors} errors",
          file=sys.stderr, flush=True)
    return {"workload": f"x <= t over {rows} rows of 20-bit values as five 4-bit lvl2 digits, "
                        f"public threshold, n0={p.n0} (6 lvl2 PBS per row: one per digit + "
                        "one combining; lvl1 result)",
            "rows": rows, "ms_per_query": ms, "errors": errors}


def run_groupby(F, ctx, sk, p, rows, reps):
    """The filter-aggregate query over a seeded synthetic table of `rows`
    rows: quantity [1, 50], price [900, 105000], discount [0, 10], tax
    [0, 8], cat1 {0, 1, 2}, cat2 {0, 1}, date [0, 2556]; WHERE date <= 2400
    GROUP BY cat1, cat2 with SUM(quantity), SUM(price * (100 - discount)),
    COUNT(*).  The encrypted part (date compared digit-wise on lvl2 against
    the public cut-off, category predicates, six group ANDs, log_rescale) is
    timed eagerly and as one replayed HIP graph; the aggregates over the
    decrypted predicates are compared with the plaintext query."""
    from cufhedb_amd import queries as Q

    rng = np.random.default_rng(41)
    cutoff = 2400
    t = {"quantity": rng.integers(1, 51, rows), "price": rng.integers(900, 105001, rows),
         "discount": rng.integers(0, 11, rows), "tax": rng.integers(0, 9, rows),
         "cat1": rng.integers(0, 3, rows), "cat2": rng.integers(0, 2, rows),
         "date": rng.integers(0, 2557, rows)}

    def enc1(v, b, seed):
        m = (np.asarray(v, np.uint64) << np.uint64(32 - b - 1)).astype(np.uint32)
        return F.DeviceBuffer.from_array(F.tlwe_encrypt_u32(seed, 0, sk.s1, m, p.alpha1))

    dd = F.DeviceBuffer.from_array(F.encrypt_digits(341, 0, sk.s2, t["date"], 3, 4, p.alpha2))
    c1, c2 = enc1(t["cat1"], 2, 342), enc1(t["cat2"], 1, 343)
    consts = [enc1([1], 2, 344), enc1([2], 2, 345), enc1([1], 1, 346)]
    scratch = Q.GroupByScratch(rows)
    run = lambda: Q.groupby_filter(ctx, dd, c1, c2, *consts, rows, cutoff,  # noqa: E731
                                   scratch=scratch)
    ok = t["date"] <= cutoff
    want = np.array([[int(np.sum(t["quantity"][m])),
                      int(np.sum(t["price"][m] * (100 - t["discount"][m]))), int(np.sum(m))]
                     for m in (ok & (t["cat1"] == a) & (t["cat2"] == b) for a, b in Q.GROUPS)],
                    np.int64)

    def errors():
        pred = Q.decrypt_predicates(scratch.out, rows, sk.s1)
        e = sum(int(np.sum(pred[g] != (ok & (t["cat1"] == a) & (t["cat2"] == b))))
                for g, (a, b) in enumerate(Q.GROUPS))
        agg = Q.group_aggregates(pred, t["quantity"], t["price"], t["discount"])
        return e, int(np.sum(agg != want))

    ms = timed_on(F, ctx, run, reps)
    err_pred, err_agg = errors()
    graph = F.Graph(ctx, run)
    ms_graph = timed_on(F, ctx, graph.launch, reps)
    gerr_pred, gerr_agg = errors()
    graph.destroy()
    scratch.free()
    for b in [dd, c1, c2] + consts:
        b.free()
    print(f"bench: group-by query {rows} rows, n0={p.n0}: {ms:.1f} ms/query "
          f"({err_pred} predicate / {err_agg} aggregate errors); graph replay {ms_graph:.1f} ms "
          f"({gerr_pred} / {gerr_agg})", file=sys.stderr, flush=True)
    return {"workload": f"SELECT cat1, cat2, SUM(quantity), SUM(price*(100-discount)), COUNT(*) "
                        f"WHERE date <= {cutoff} GROUP BY cat1, cat2 over {rows} seeded rows, "
                        f"n0={p.n0}: date as three 4-bit lvl2 digits vs the public cut-off "
                        "(4 lvl2 PBS), 3 lvl1 category compares, 10 lvl1 ANDs, 6 log_rescales "
                        "per row; aggregates over the decrypted predicates",
            "rows": rows, "ms_per_query": ms, "ms_per_query_graph": ms_graph,
            "predicate_errors": err_pred, "aggregate_errors": err_agg,
            "predicate_errors_graph": gerr_pred, "aggregate_errors_graph": gerr_agg,
            "aggregates": {f"{a},{b}": want[g].tolist() for g, (a, b) in enumerate(Q.GROUPS)}}


def run_queries(F, ctx, sk, p, rows, reps):
    """Encrypted query pipelines, each timed with HIP events on the context
    stream over `reps` runs after one untimed run (which also sizes the
    operator scratch); inputs resident on the device, results decrypted and
    compared with the plaintext query."""
    from cufhedb_amd import queries as Q

    L_ = F.lib()
    rng = np.random.default_rng(13)
    res = {"preset": f"n0={p.n0} (reference parameter set)"}

    def timed(fn):
        return timed_on(F, ctx, fn, reps)

    # lvl2 PBS throughput (the chains' dominant operation): batch 4096
    B2 = 4096
    c0 = F.tlwe_encrypt_u32(303, 0, sk.s0, (rng.integers(0, 8, B2) << 28).astype(np.uint32),
                            p.alpha0)
    d0 = F.DeviceBuffer.from_array(c0)
    tv2 = F.DeviceBuffer.from_array(np.full(2048, 1 << 61, np.uint64))
    o2 = F.DeviceBuffer(B2 * 2049 * 8)
    ms2 = timed(lambda: F.check(L_.fhe_pbs_lvl02_dev(ctx.h, d0.ptr, tv2.ptr, 0, o2.ptr, B2, None)))
    res["lvl2_pbs"] = {"workload": f"lvl2 PBS (N=2048, l=4, Bgbit=9, 64-bit torus), batch {B2}",
                       "ms_per_step": ms2, "pbs_per_s": B2 / (ms2 / 1e3)}
    print(f"bench: lvl2 PBS batch {B2}: {ms2:.1f} ms, {B2 / (ms2 / 1e3):.0f} PBS/s",
          file=sys.stderr, flush=True)
    for b in (d0, tv2, o2):
        b.free()

    # range filter x <= t, 20-bit values on the 64-bit torus, shared threshold
    bits = 20
    x = rng.integers(0, 1 << bits, rows)
    t = int(rng.integers(0, 1 << bits))
    sc = np.uint64(64 - bits - 1)
    dx = F.DeviceBuffer.from_array(
        F.tlwe_encrypt_u64(301, 0, sk.s2, x.astype(np.uint64) << sc, p.alpha2))
    dt = F.DeviceBuffer.from_array(
        F.tlwe_encrypt_u64(302, 0, sk.s2, np.array([t], np.uint64) << sc, p.alpha2))
    out = F.DeviceBuffer(rows * (N + 1) * 4)
    ms = timed(lambda: Q.range_filter(ctx, dx, dt, rows, bits, out_dev=out))
    ph = F.tlwe_phase_u32(out.to_array(np.uint32, (rows, N + 1)), sk.s1).view(np.int32)
    errors = int(np.sum((ph > 0) != (x <= t)))
    res["range_filter"] = {
        "workload": f"x <= t over {rows} rows of {bits}-bit lvl2 values, one shared encrypted "
                    "threshold (HomMSB chain: 6 lvl2 + 3 lvl1 PBS per row)",
        "rows": rows, "ms_per_query": ms, "errors": errors}
    print(f"bench: range filter {rows} rows: {ms:.1f} ms/query, {errors} errors",
          file=sys.stderr, flush=True)
    for b in (dx, dt, out):
        b.free()
    res["compare_digits"] = run_compare_digits(F, ctx, sk, p, rows, reps)

    # TPC-H Q1 filter: shipdate <= date, 4 (returnflag, linestatus) groups
    date_bits = 9
    rf = rng.integers(0, 2, rows)
    ls = rng.integers(0, 2, rows)
    date = rng.integers(0, 1 << date_bits, rows)
    qty = rng.integers(0, 256, rows)
    thr = int(rng.integers(0, 1 << date_bits))

    def enc1(v, b, seed):
        m = (np.asarray(v, np.uint64) << np.uint64(32 - b - 1)).astype(np.uint32)
        return F.DeviceBuffer.from_array(F.tlwe_encrypt_u32(seed, 0, sk.s1, m, p.alpha1))

    cols = [enc1(date, date_bits, 311), enc1(rf, 1, 312), enc1(ls, 1, 313)]
    dthr, one = enc1([thr], date_bits, 314), enc1([1], 1, 315)
    scratch = Q.Q1Scratch(rows)
    ms = timed(lambda: Q.tpch_q1_filter(ctx, cols[0], cols[1], cols[2], dthr, one, rows,
                                        scratch=scratch))
    pred = Q.decrypt_predicates(scratch.out, rows, sk.s1)
    ok = date <= thr
    errors = 0
    for g, (a, b) in enumerate(((0, 0), (0, 1), (1, 0), (1, 1))):
        want = ok & (rf == a) & (ls == b)
        errors += int(np.sum(pred[g] != want))
        errors += int(int(np.sum(qty * pred[g])) != int(np.sum(qty[want])))
    # the same pipeline captured once into a HIP graph and replayed
    graph = F.Graph(ctx, lambda: Q.tpch_q1_filter(ctx, cols[0], cols[1], cols[2], dthr, one,
                                                  rows, scratch=scratch))
    ms_graph = timed(graph.launch)
    pred = Q.decrypt_predicates(scratch.out, rows, sk.s1)
    errors_graph = sum(int(np.sum(pred[g] != (ok & (rf == a) & (ls == b))))
                       for g, (a, b) in enumerate(((0, 0), (0, 1), (1, 0), (1, 1))))
    graph.destroy()
    # small batches, where host launch overhead shows: eager calls vs graph
    small = 256
    sscr = Q.Q1Scratch(small)
    run_small = lambda: Q.tpch_q1_filter(ctx, cols[0], cols[1], cols[2], dthr, one, small,  # noqa
                                         scratch=sscr)
    ms_small = timed_on(F, ctx, run_small, 20)
    gsmall = F.Graph(ctx, run_small)
    ms_small_graph = timed_on(F, ctx, gsmall.launch, 20)
    gsmall.destroy()
    sscr.free()
    res["tpch_q1_filter"] = {
        "workload": f"TPC-H Q1 filter on {rows} lvl1 rows: shipdate <= date (9 bit), "
                    "4 (returnflag, linestatus) groups, log_rescale; SUM(qty)/COUNT after "
                    "decryption",
        "rows": rows, "ms_per_query": ms, "errors": errors,
        "ms_per_query_graph": ms_graph, "errors_graph": errors_graph,
        "small_rows": small, "small_ms_eager": ms_small, "small_ms_graph": ms_small_graph}
    print(f"bench: TPC-H Q1 filter {rows} rows: {ms:.1f} ms/query, {errors} errors; "
          f"graph replay {ms_graph:.1f} ms, {errors_graph} errors; {small} rows: eager "
          f"{ms_small:.2f} ms, graph {ms_small_graph:.2f} ms", file=sys.stderr, flush=True)
    scratch.free()
    for b in cols + [dthr, one]:
        b.free()
    return res


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--batch", type=int, default=8192)
    ap.add_argument("--preset", choices=["cfg636", "ref672"], default="cfg636")
    ap.add_argument("--variant", choices=["fp64", "mfma_split", "both"], default="both",
                    help="lvl1 PBS kernel variant(s) to time; 'both' reports each and takes the "
                         "faster for the headline value")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-query", action="store_true",
                    help="skip the encrypted-query pipelines (range filter, TPC-H Q1 filter)")
    ap.add_argument("--query-rows", type=int, default=1 << 14)
    ap.add_argument("--query-reps", type=int, default=2)
    ap.add_argument("--mixed", type=int, default=200, metavar="NBATCHES",
                    help="also run the mixed lvl1-PBS / lvl2-compare batch stream of this many "
                         "batches (sizes lognormal around 2048 clipped to [256, 65536], 70%% "
                         "lvl1) through the scheduler; 0 skips it")
    ap.add_argument("--mixed-all", action="store_true",
                    help="also run the stream one call per batch, and digit-wise at n0 = 636")
    ap.add_argument("--calib-copy-mib", type=int, default=0,
                    help="also run one device-to-device copy of this many MiB (a plain copy "
                         "kernel of known size, to scale rocprofv3 FETCH_SIZE / WRITE_SIZE)")
    args = ap.parse_args()

    if args.gpus != 1:
        print(f"bench.py: this build runs on one GPU; --gpus {args.gpus} is not supported "
              "(the path would shard by ciphertext: every GPU holding the keys, B/G "
              "ciphertexts each, results gathered afterwards)",
              file=sys.stderr)
        sys.exit(2)

    import cufhedb_amd as F

    which = F.PRESET_CFG636 if args.preset == "cfg636" else F.PRESET_REF672
    p = F.preset(which)
    sk = F.SecretKeys(p, 20261202)
    bk = F.keygen_bk_lvl01(sk, 20261203)
    ctx = F.Context(p, 0)
    ctx.load_bk(1, bk, F.BK_INT)

    B = args.batch
    rng = np.random.default_rng(11)
    m = rng.integers(0, 8, B)
    lut = rng.integers(0, 8, 8)
    tv = z8_testvector(lut)
    c0 = F.tlwe_encrypt_u32(20261204, 0, sk.s0, (m << 28).astype(np.uint32), p.alpha0)
    d_in = F.DeviceBuffer.from_array(c0)
    d_tv = F.DeviceBuffer.from_array(tv)
    d_out = F.DeviceBuffer(B * (N + 1) * 4)
    L_ = F.lib()

    def step():
        F.check(L_.fhe_pbs_lvl01_dev(ctx.h, d_in.ptr, d_tv.ptr, 0, d_out.ptr, B, None))

    if args.calib_copy_mib:
        nb = args.calib_copy_mib << 20
        src, dst = F.DeviceBuffer(nb), F.DeviceBuffer(nb)
        F.check(L_.fhe_memcpy_d2d(dst.ptr, src.ptr, nb))
        F.check(L_.fhe_device_sync())
        src.free()
        dst.free()

    codes = {"fp64": F.PBS_FP64, "mfma_split": F.PBS_MFMA_SPLIT}
    names = ["fp64", "mfma_split"] if args.variant == "both" else [args.variant]
    variants = {}
    for name in names:
        try:
            ctx.set_pbs_variant(codes[name])
        except F.FheError as e:
            variants[name] = {"unsupported": str(e)}
            print(f"bench: {name}: {e}", file=sys.stderr, flush=True)
            continue
        for _ in range(args.warmup):
            step()
        ctx.sync()
        print(f"bench: {name}: warmup done ({args.warmup} x {B} PBS)", file=sys.stderr,
              flush=True)
        F.check(L_.fhe_timer_start(ctx.h, None))
        for _ in range(args.steps):
            step()
        ms = ctypes.c_float()
        F.check(L_.fhe_timer_stop(ctx.h, None, ctypes.byref(ms)))
        total_ms = float(ms.value)
        out = d_out.to_array(np.uint32, (B, N + 1))
        ph = F.tlwe_phase_u32(out, sk.s1).view(np.int32).astype(np.int64)
        dec = np.round(ph / (1 << 28)).astype(np.int64) % 16
        err = ph - lut[m] * (1 << 28)
        # |phase error| per octave, in 2^-32 torus units (decision margin 2^27)
        edges = [0] + [1 << j for j in range(18, 28)] + [1 << 62]
        hist = np.histogram(np.abs(err), bins=edges)[0]
        labels = ["<2^18"] + [f"2^{j}" for j in range(18, 27)] + [">=2^27"]
        variants[name] = {
            "ms_per_step": total_ms / args.steps,
            "pbs_per_s": B * args.steps / (total_ms / 1e3),
            "decrypt_failures": int(np.sum(dec != lut[m])),
            "phase_error_std_log2": float(np.log2(np.std(err))),
            "phase_error_hist": {lab: int(c) for lab, c in zip(labels, hist)},
        }
        if name == "mfma_split":
            # matrix-core work actually issued (utilisation diagnostic, not the
            # roofline figure): per forward transform 4 v_mfma_f32_32x32x16_f16
            # (32768 flops each) and 24 v_mfma_f32_16x16x32_f16 (16384 each),
            # six transforms per CMUX step
            mf = p.n0 * 6 * (4 * 32768 + 24 * 16384)
            rate = variants[name]["pbs_per_s"] * mf / 1e12
            variants[name].update({"mfma_flops_per_pbs": mf, "mfma_tflops": rate,
                                   "mfma_frac_of_fp16_dense_peak": rate / 2500.0})
        print(f"bench: {name}: timed {args.steps} steps, {total_ms / args.steps:.3f} ms/step, "
              f"{variants[name]['decrypt_failures']} decryption failures", file=sys.stderr,
              flush=True)
    # the headline is the fastest variant that decrypts every output
    ran = [k for k in variants if "pbs_per_s" in variants[k]]
    exact = [k for k in ran if variants[k]["decrypt_failures"] == 0] or ran
    best = max(exact, key=lambda k: variants[k]["pbs_per_s"])
    ms_per_step = variants[best]["ms_per_step"]
    value = variants[best]["pbs_per_s"]
    failures = variants[best]["decrypt_failures"]
    if len(ran) == 2:
        variants["mfma_split_over_fp64"] = (variants["mfma_split"]["pbs_per_s"] /
                                            variants["fp64"]["pbs_per_s"])
    ctx.set_pbs_variant(codes[best])

    fl = flops_per_pbs(p.n0)
    achieved = fl * B / (ms_per_step / 1e3) / 1e12
    roofline = {
        # compute-bound: the FP64 VALU (MI355X's FP64 vector peak equals its
        # FP64 matrix peak, 78.6 TFLOP/s; no matrix instruction is issued)
        "bound": "mfma",
        "compute_unit": "fp64 valu" if best == "fp64" else "fp16 mfma + fp32/fp64 valu",
        "achieved": achieved,
        "peak": PEAK_FP64_TFLOPS,
        "unit": "TFLOP/s",
        "frac": achieved / PEAK_FP64_TFLOPS,
        "traffic": load_traffic(best, args.preset, B),
        "kernel": ("k_blind_rotate1 (FP64 VALU; MI355X FP64 vector == FP64 matrix peak)"
                   if best == "fp64" else
                   "k_blind_rotate1_mfma (fp16 MFMA forward transforms; bound by its FP64/FP32 "
                   "VALU work, priced at the FP64 peak)"),
        "flops_per_pbs": fl,
    }
    # the same kernel against ceilings measured on this device (FP64 FMA
    # micro-kernel; streaming copy), next to the published peak above
    fp64_meas, copy_meas = ctypes.c_double(), ctypes.c_double()
    F.check(L_.fhe_measure_peaks(ctx.h, ctypes.byref(fp64_meas), ctypes.byref(copy_meas)))
    roofline["measured"] = {"fp64_fma_tflops": fp64_meas.value,
                            "frac": achieved / fp64_meas.value,
                            "copy_gbs": copy_meas.value}
    print(f"bench: measured FP64 FMA {fp64_meas.value:.1f} TFLOP/s, copy "
          f"{copy_meas.value:.0f} GB/s", file=sys.stderr, flush=True)
    res = {
        "metric": METRIC,
        "value": value,
        "unit": "PBS/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_per_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64" if best == "fp64" else "f16-split/f32/f64",
        "data": "synthetic (seeded keys and Z_8 plaintexts, random 8-entry LUT)",
        "config": {
            "workload": f"lvl1 PBS (BlindRotate+SampleExtract), batch {B}, n0={p.n0}, "
                        f"N=1024 k=1 l=3 Bgbit=6, {best}",
            "batch": B,
            "n0": int(p.n0),
            "variant": best,
        },
        "roofline": roofline,
        "variants": variants,
        "decrypt_failures": failures,
        "device": F.device_name(),
    }
    ctx.close()
    res["queries"] = None
    # the headline kernel on the reference's parameter set (n0 = 672), for a
    # like-for-like comparison with the CPU baseline (compiled TFHEpp, whose
    # n0 is fixed at 672)
    gpu672 = None
    gates672 = None
    if not args.no_query or args.mixed or not args.no_cpu_baseline:
        octx, osk, op = operator_context(F)
        gpu672 = pbs_lvl01_rate(F, octx, osk, op, B, 5)
        if not args.no_cpu_baseline:
            gates672 = gate_and_iks_rates(F, octx, osk, op, B, 5, min(16, os.cpu_count() or 1))
    if not args.no_query or args.mixed:
        res["autotune"] = autotune(F, octx)
        if not args.no_query:
            res["queries"] = run_queries(F, octx, osk, op, args.query_rows, args.query_reps)
        if args.mixed:
            from cufhedb_amd import mixed
            plan = mixed.make_plan(2026, args.mixed)
            sizes = [b for _, b in plan]
            _, coal = mixed.run_coalesced(octx, osk, op, plan)
            res["mixed_stream"] = {
                "workload": f"{len(plan)} batches, {sum(sizes)} rows, sizes lognormal around "
                            "2048 clipped to [256, 65536], 70% lvl1 Z_8 LUT PBS / 30% lvl2 "
                            "20-bit x <= t (HomMSB chain), n0=672, all submitted at once to "
                            "the scheduler; latency from the flush start",
                "coalesced": coal}
            print(f"bench: mixed stream, scheduler: {coal}", file=sys.stderr, flush=True)
            if args.mixed_all:
                _, seq = mixed.run(octx, osk, op, plan)
                res["mixed_stream"]["sequential"] = seq
                print(f"bench: mixed stream, one call per batch: {seq}", file=sys.stderr,
                      flush=True)
    if gpu672 is not None:
        octx.close()
        if args.mixed and args.mixed_all:
            # the same plan at n0 = 636 with the comparisons digit-wise
            # against public thresholds (the HomMSB chain needs n0 = 672)
            octx, osk, op = operator_context(F, F.PRESET_CFG636)
            if "autotune" in res:
                apply_tuning(F, octx, res["autotune"])
            _, dig = mixed.run(octx, osk, op, plan, compare="digits")
            res["mixed_stream"]["sequential_digits_n636"] = dig
            print(f"bench: mixed stream, digit-wise compares at n0=636: {dig}", file=sys.stderr,
                  flush=True)
            octx.close()
        if not args.no_query:
            # the 20-bit comparison workload at its own parameter set, n0 = 636
            octx, osk, op = operator_context(F, F.PRESET_CFG636)
            apply_tuning(F, octx, res["autotune"])
            res["queries"]["compare_digits_n636"] = run_compare_digits(
                F, octx, osk, op, args.query_rows, args.query_reps)
            res["queries"]["groupby_n636"] = run_groupby(F, octx, osk, op, args.query_rows,
                                                         args.query_reps)
            octx.close()
    if not args.no_cpu_baseline:
        threads = min(16, os.cpu_count() or 1)
        res["cpu_baseline"] = cpu_baseline(threads)
        if gpu672 is not None and res["cpu_baseline"]["kind"] == "reference":
            # both at n0 = 672: GPU FP64 kernel vs compiled TFHEpp on the host
            res["cpu_baseline"]["gpu_same_params"] = dict(
                gpu672, gpu_over_cpu=gpu672["pbs_per_s"] / res["cpu_baseline"]["value"])
        if gates672 is not None:
            res["cpu_baseline"]["gate_and_key_switch"] = gates672
    else:
        res["cpu_baseline"] = None
    print(json.dumps(res))


if __name__ == "__main__":
    main()
