"""Benchmark of the MI355X CKKS key-switch hot path.

Headline (BASELINE.json "metric", configs[1]): batched NTT + INTT of one
ciphertext, 2 polynomials x 32 RNS limbs, N = 2^16, 32 distinct 30-bit
primes = 1 mod 2^17, limb-major. One step = forward NTT of all 64 limbs
followed by the inverse NTT (128 limb-transforms). value = limb-transforms/s
with inputs resident in HBM; the input/output buffers rotate over a set
larger than the 256 MB MALL so the timed traffic comes from HBM.
Consecutive steps are independent ciphertexts and alternate over three HIP
streams (a buffer set always on the same stream), so one step's load phase
runs beside another's butterflies; the one-stream step time, the latency
of one batch, is reported next to it.

The same JSON line carries the other two parts of the metric: the HMult
key-switch time at config 4 (L = 24, dnum = 3, alpha = 8, merged
ModDown+Rescale; also without rescale followed by a separate Rescale, and
independent HMults over three streams) and the config-3 BConv time, all
measured with HIP events, the time of a config-5-shaped hoisted BSGS linear
transform, plus the roofline of the NTT and the CPU baseline (the oracle's
scalar Montgomery NTT on this host, bounded sample).

    python bench.py [--gpus 1] [--steps K] [--warmup W]
"""
import argparse
import ctypes
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "cheddar-fhe_amd", "python"))

HBM_PEAK_GBS = 8000.0
INT8_PEAK_TOPS = 5000.0     # dense int8 MFMA, MI355X
# config 3 BConv: 8 limbs in + 40 limbs out; useful int8 operations of the
# byte-split product (16 byte products per 32 x 32-bit product, 2 ops each)
BCONV_BYTES = 48 * 4 * (1 << 16)
BCONV_INT8_OPS = 2 * 16 * (1 << 16) * 8 * 40
# its measured HBM bytes per launch (profiles/bconv_config3_traffic.md:
# FETCH_SIZE 1101.0 KiB x 2 + WRITE_SIZE 10240.0 KiB)
BCONV_TRAFFIC = 12741632
# config 4 HMult compulsory bytes: 4 x 24 input limbs, 3 x 2 x 32 key limbs,
# 2 x 23 output limbs
HMULT_BYTES = (96 + 192 + 46) * 4 * (1 << 16)
# its measured HBM bytes per HMult, the sum over its 5 launches
# (profiles/hmult_switch_config4_traffic.md, one row per launch)
HMULT_SWITCH_TRAFFIC = 27440128 + 26079232 + 134737536 + 17345536 + 44419072
# and of the eight-launch form before it (profiles/hmult_config4_traffic.md)
HMULT_TRAFFIC = (25288704 + 12904384 + 25421824 + 38169344 + 128323392 +
                 9696448 + 16902144 + 48662528)
N = 1 << 16
LIMB_BYTES = 4 * N
# one limb-transform moves one limb in and one limb out (algorithmic bytes)
LIMB_TRANSFORM_BYTES = 2 * LIMB_BYTES
MALL_BYTES = 256 << 20
# calibration copy: 1 GiB each way, far beyond L2 and the 256 MiB MALL
COPY_BYTES = 1 << 30
# the headline's consecutive steps alternate over this many streams
NTT_STREAMS = 3


def ntt_sets():
    """buffer sets of the headline loop: more than twice the MALL per role,
    a multiple of NTT_STREAMS so that set j is only ever used on stream
    j % NTT_STREAMS"""
    n = max(4, (2 * MALL_BYTES) // (2 * 32 * LIMB_BYTES) + 1)
    return (n + NTT_STREAMS - 1) // NTT_STREAMS * NTT_STREAMS


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--no-cpu", action="store_true",
                    help="skip the CPU-baseline leg")
    ap.add_argument("--only", choices=["ntt_fwd", "ntt_inv", "ntt_inv_1p",
                                       "ntt_step",
                                       "hmult",
                                       "hmult_cold", "hmult_separate",
                                       "hmult_levels", "hrot",
                                       "bconv", "bconv_cold",
                                       "copy", "hoist"],
                    help="run only this workload's timed loop (for "
                         "profiling); prints its average time")
    return ap.parse_args()


def event_time_ms(fn, iters, stream):
    import torch
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    start.record(stream)
    for i in range(iters):
        fn(i)
    end.record(stream)
    end.synchronize()
    return start.elapsed_time(end)


def bench_ntt(chd, steps, warmup):
    import numpy as np
    import torch
    from chd_primes import ntt_primes
    primes = ntt_primes(30, 32)
    plan = chd.NttPlan(primes)
    nsets = ntt_sets()
    rng = np.random.default_rng(0xC0FFEE02)
    host = np.stack([np.stack([rng.integers(0, p, N, dtype=np.uint64)
                               for p in primes]) for _ in range(2)])
    base = torch.from_numpy(host.astype(np.uint32).view(np.int32)).cuda()
    srcs = [base.clone() for _ in range(nsets)]
    dsts = [torch.empty_like(base) for _ in range(nsets)]
    stream = torch.cuda.current_stream()
    sp = ctypes.c_void_p(stream.cuda_stream)

    streams = [torch.cuda.Stream() for _ in range(NTT_STREAMS)]
    sps = [ctypes.c_void_p(x.cuda_stream) for x in streams]

    def step_on(i, p, two_pass=False):
        s, d = srcs[i % nsets], dsts[i % nsets]
        plan.forward(d, s, 32, 2, stream=p, two_pass=two_pass)
        plan.inverse(s, d, 32, 2, mont_conv=False, stream=p)

    # Per-direction timings (reported, and the forward one is the roofline's)
    # come first, over at least 200 calls each: back to back they keep the
    # GPU busy for ~10 ms, so the headline loop below starts at sustained
    # clocks (its W warmup steps alone take 0.2 ms at the driver's W = 5).
    # The inverse restores the sources the forward read (mont_conv=False).
    sub = max(steps, 200)
    def fwd(i):
        plan.forward(dsts[i % nsets], srcs[i % nsets], 32, 2, stream=sp)
    fwd_ms = event_time_ms(fwd, sub, stream) / sub
    inv_ms = event_time_ms(
        lambda i: plan.inverse(srcs[i % nsets], dsts[i % nsets], 32, 2,
                               mont_conv=False, stream=sp), sub,
        stream) / sub
    # the single-pass inverse (one HBM read and write per limb), for
    # comparison: the same results, not used by the headline loop
    inv1_ms = event_time_ms(
        lambda i: plan.inverse(srcs[i % nsets], dsts[i % nsets], 32, 2,
                               mont_conv=False, stream=sp,
                               single_pass=True), sub,
        stream) / sub
    # the forward on the two-pass kernels (chd_ntt_forward_two_pass)
    fwd2_ms = event_time_ms(
        lambda i: plan.forward(dsts[i % nsets], srcs[i % nsets], 32, 2,
                               stream=sp, two_pass=True), sub, stream) / sub
    # warm (MALL-resident) figure on one buffer set
    warm_ms = event_time_ms(lambda i: plan.forward(dsts[0], srcs[0], 32, 2,
                                                   stream=sp), sub,
                            stream) / sub
    # one step at a time on one stream: the latency of one batch
    one_ms = event_time_ms(lambda i: step_on(i, sp), sub, stream) / sub
    # the headline: W warmup steps, then exactly K timed steps, step i on
    # stream i % NTT_STREAMS (set i % nsets, so a set never changes stream)
    for i in range(warmup):
        step_on(i, sps[i % NTT_STREAMS])
    torch.cuda.synchronize()
    # an event at the start and the end of each stream's share; the timed
    # span runs from the earliest start to the latest end (no cross-stream
    # waits added to the loop)
    starts = [torch.cuda.Event(enable_timing=True) for _ in streams]
    ends = [torch.cuda.Event(enable_timing=True) for _ in streams]
    for ev, x in zip(starts, streams):
        ev.record(x)
    for i in range(steps):
        step_on(i, sps[i % NTT_STREAMS])
    for ev, x in zip(ends, streams):
        ev.record(x)
    torch.cuda.synchronize()

    def span(starts, ends):
        t0 = starts[0]
        return (max(t0.elapsed_time(ev) for ev in ends) -
                min([0.0] + [t0.elapsed_time(ev) for ev in starts[1:]]))
    ms = span(starts, ends)
    # the same loop with the forward on the two-pass kernels, after the
    # headline (reported beside it, not the headline)
    for ev, x in zip(starts, streams):
        ev.record(x)
    for i in range(steps):
        step_on(i, sps[i % NTT_STREAMS], two_pass=True)
    for ev, x in zip(ends, streams):
        ev.record(x)
    torch.cuda.synchronize()
    ms2 = span(starts, ends)
    # the inverse with mont_conv=False returns the input: check it stayed put
    ok = all(torch.equal(srcs[i], base) for i in range(nsets))
    return ms, fwd_ms, inv_ms, warm_ms, one_ms, ok, inv1_ms, fwd2_ms, ms2


def _config4_context(chd):
    from chd_primes import ntt_primes
    main, aux = ntt_primes(30, 24), ntt_primes(31, 8)
    param = chd.Param(main, aux, [(i, 0) for i in range(1, 25)])
    return main, aux, chd.Context(param)


def bench_hmult(chd, iters=20, cold=False, separate=False):
    """config 4: HMult with merged rescale at L = 24. warm: the same inputs
    and key every step (working set resident in the 256 MB MALL); cold:
    steps rotate over distinct input/key sets spanning more than twice the
    MALL, so inputs and keys come from HBM. separate: HMult without rescale
    followed by a separate Rescale (the reference's other form)"""
    import numpy as np
    import torch
    main, aux, ctx = _config4_context(chd)
    rng = np.random.default_rng(0xC0FFEE04)

    def limbs(primes):
        a = np.stack([rng.integers(0, p, N, dtype=np.uint64) for p in primes])
        return torch.from_numpy(a.astype(np.uint32).view(np.int32)).cuda()
    set_bytes = (4 * 24 + 6 * 32) * LIMB_BYTES
    nsets = (2 * MALL_BYTES) // set_bytes + 2 if cold else 1
    base = [limbs(main) for _ in range(4)] + [limbs(main + aux)
                                              for _ in range(6)]
    sets = [base] + [[t.clone() for t in base] for _ in range(nsets - 1)]
    res = (torch.empty(23, N, dtype=torch.int32, device="cuda"),
           torch.empty(23, N, dtype=torch.int32, device="cuda"))
    full = (torch.empty(24, N, dtype=torch.int32, device="cuda"),
            torch.empty(24, N, dtype=torch.int32, device="cuda"))
    stream = torch.cuda.current_stream()
    sp = ctypes.c_void_p(stream.cuda_stream)

    def run(i):
        t = sets[i % nsets]
        if separate:
            ctx.hmult(23, full, (t[0], t[1]), (t[2], t[3]), t[4:7], t[7:10],
                      rescale=False, stream=sp)
            ctx.rescale(23, res, full, stream=sp)
        else:
            ctx.hmult(23, res, (t[0], t[1]), (t[2], t[3]), t[4:7], t[7:10],
                      rescale=True, stream=sp)
    for i in range(3):
        run(i)
    torch.cuda.synchronize()
    return event_time_ms(run, iters, stream) / iters, nsets * set_bytes


def bench_hrot(chd, iters=20):
    """config 4: HRot by 1234 slots at L = 24 (MultKey, whose key
    accumulation adds P times bx, then Permute), the same input and key
    every step"""
    import numpy as np
    import torch
    main, aux, ctx = _config4_context(chd)
    rng = np.random.default_rng(0xC0FFEE06)

    def limbs(primes):
        a = np.stack([rng.integers(0, p, N, dtype=np.uint64) for p in primes])
        return torch.from_numpy(a.astype(np.uint32).view(np.int32)).cuda()
    a = (limbs(main), limbs(main))
    kb = [limbs(main + aux) for _ in range(3)]
    ka = [limbs(main + aux) for _ in range(3)]
    res = (torch.empty(24, N, dtype=torch.int32, device="cuda"),
           torch.empty(24, N, dtype=torch.int32, device="cuda"))
    stream = torch.cuda.current_stream()
    sp = ctypes.c_void_p(stream.cuda_stream)

    def run(i):
        ctx.hrot(23, res, a, kb, ka, 1234, stream=sp)
    for i in range(3):
        run(i)
    torch.cuda.synchronize()
    return event_time_ms(run, iters, stream) / iters


def bench_hmult_levels(chd, levels=(4, 8, 12, 16, 20, 24), iters=50):
    """HMult (merged rescale) of the config-4 chain at several levels: L q
    limbs in, L - 1 out, ceil(L / 8) of the key's 3 dnum groups in use, the
    same key and inputs every step (warm). Returns {L: microseconds}."""
    import numpy as np
    import torch
    main, aux, ctx = _config4_context(chd)
    rng = np.random.default_rng(0xC0FFEE24)

    def limbs(primes):
        a = np.stack([rng.integers(0, p, N, dtype=np.uint64) for p in primes])
        return torch.from_numpy(a.astype(np.uint32).view(np.int32)).cuda()
    kb = [limbs(main + aux) for _ in range(3)]
    ka = [limbs(main + aux) for _ in range(3)]
    stream = torch.cuda.current_stream()
    sp = ctypes.c_void_p(stream.cuda_stream)
    out = {}
    for L in levels:
        x = [limbs(main[:L]) for _ in range(4)]
        res = (torch.empty(L - 1, N, dtype=torch.int32, device="cuda"),
               torch.empty(L - 1, N, dtype=torch.int32, device="cuda"))
        def run(i):
            ctx.hmult(L - 1, res, (x[0], x[1]), (x[2], x[3]), kb, ka,
                      rescale=True, stream=sp)
        for i in range(3):
            run(i)
        torch.cuda.synchronize()
        out[L] = event_time_ms(run, iters, stream) / iters * 1e3
    return out


def bench_hmult_streams(chd, iters=150, nstreams=NTT_STREAMS):
    """config 4 throughput: independent HMults (merged rescale) alternating
    over nstreams HIP streams, one Context per stream (a Context serialises
    its calls on its key-switch arena) and one input/key set per stream.
    Returns microseconds per HMult over the span from the earliest
    per-stream start event to the latest end event."""
    import numpy as np
    import torch
    ctxs = [_config4_context(chd) for _ in range(nstreams)]
    main, aux = ctxs[0][0], ctxs[0][1]
    rng = np.random.default_rng(0xC0FFEE14)

    def limbs(primes):
        a = np.stack([rng.integers(0, p, N, dtype=np.uint64) for p in primes])
        return torch.from_numpy(a.astype(np.uint32).view(np.int32)).cuda()
    sets = [[limbs(main) for _ in range(4)] + [limbs(main + aux)
                                               for _ in range(6)]
            for _ in range(nstreams)]
    res = [(torch.empty(23, N, dtype=torch.int32, device="cuda"),
            torch.empty(23, N, dtype=torch.int32, device="cuda"))
           for _ in range(nstreams)]
    streams = [torch.cuda.Stream() for _ in range(nstreams)]
    sps = [ctypes.c_void_p(x.cuda_stream) for x in streams]

    def run(i):
        k = i % nstreams
        t = sets[k]
        ctxs[k][2].hmult(23, res[k], (t[0], t[1]), (t[2], t[3]), t[4:7],
                         t[7:10], rescale=True, stream=sps[k])
    for i in range(3 * nstreams):
        run(i)
    torch.cuda.synchronize()
    starts = [torch.cuda.Event(enable_timing=True) for _ in streams]
    ends = [torch.cuda.Event(enable_timing=True) for _ in streams]
    for ev, x in zip(starts, streams):
        ev.record(x)
    for i in range(iters):
        run(i)
    for ev, x in zip(ends, streams):
        ev.record(x)
    torch.cuda.synchronize()
    t0 = starts[0]
    span = (max(t0.elapsed_time(e) for e in ends) -
            min(t0.elapsed_time(s) for s in starts))
    return span / iters * 1e3


def bench_hoist(chd, iters=5):
    """config 5: the 768 x 768 BSGS linear transform (28 baby steps, 28
    giant steps 28 k, 54 rotation keys) on one ciphertext at L = 20 of the
    config-4 chain, double hoisting. The 768 plaintexts are the generalised
    diagonals of a seeded W ~ N(0, 0.02), each rotated by its giant step,
    encoded by the library at scale 2^30 into 2^15 slots with the alpha aux
    primes (the reference's message constructor); ciphertext and keys are
    seeded uniform residues."""
    import numpy as np
    import torch
    main, aux, ctx = _config4_context(chd)
    L, level, dim, slots = 20, 19, 768, 1 << 15
    r = np.random.default_rng(0xC0FFEE05)
    W = r.normal(0.0, 0.02, (dim, dim))
    bs = list(range(28))
    gs = [28 * k for k in range(28)]
    rows = np.arange(dim)
    msgs = {}
    for g in gs:
        for b in bs:
            if g + b < dim:
                diag = np.zeros(slots)
                diag[:dim] = W[rows, (rows + g + b) % dim]
                msgs[(g, b)] = np.roll(diag, g).astype(np.complex128)
    h = chd.Hoist.from_messages(ctx, level, 2.0 ** 30, gs, bs, msgs)
    del msgs
    gen = torch.Generator(device="cuda")
    gen.manual_seed(0xC0FFEE05)

    def limbs(n):
        return torch.randint(0, 1 << 29, (n, N), dtype=torch.int32,
                             device="cuda", generator=gen)
    rots = h.required_rotations()
    keys = {rot: ([limbs(32) for _ in range(3)], [limbs(32) for _ in range(3)])
            for rot in rots}
    ct = (limbs(L), limbs(L))
    res = (torch.empty(L - 1, N, dtype=torch.int32, device="cuda"),
           torch.empty(L - 1, N, dtype=torch.int32, device="cuda"))
    stream = torch.cuda.current_stream()
    sp = ctypes.c_void_p(stream.cuda_stream)
    for _ in range(2):
        h.run(res, ct, keys, stream=sp)
    torch.cuda.synchronize()
    ms = event_time_ms(lambda i: h.run(res, ct, keys, stream=sp), iters,
                       stream) / iters
    # bytes every evaluation has to read once: the plaintexts (L + alpha
    # limbs each) and, per key switch (27 baby + 27 giant), the key's
    # dnum groups over L + alpha limbs
    assert len(rots) == 54
    compulsory = (dim * (L + 8) + len(rots) * 3 * 2 * (L + 8)) * LIMB_BYTES
    return ms, compulsory


def bench_bconv(chd, iters=50, cold=False):
    """config 3: BConv 8 -> 40 limbs. cold: steps rotate over distinct
    source/destination sets spanning more than twice the MALL"""
    import numpy as np
    import torch
    from chd_primes import ntt_primes
    src_p, dst_p = ntt_primes(30, 8), ntt_primes(31, 40)
    plan = chd.BconvPlan(src_p, dst_p)
    rng = np.random.default_rng(0xC0FFEE03)
    x = np.stack([rng.integers(-((p - 1) // 2), (p - 1) // 2 + 1, N)
                  for p in src_p]).astype(np.int32)
    set_bytes = 48 * LIMB_BYTES
    nsets = (2 * MALL_BYTES) // set_bytes + 2 if cold else 1
    src0 = torch.from_numpy(x).cuda()
    srcs = [src0] + [src0.clone() for _ in range(nsets - 1)]
    dsts = [torch.empty(40, N, dtype=torch.int32, device="cuda")
            for _ in range(nsets)]
    stream = torch.cuda.current_stream()
    sp = ctypes.c_void_p(stream.cuda_stream)

    def run(i):
        plan.apply(dsts[i % nsets], srcs[i % nsets], stream=sp)
    for i in range(3):
        run(i)
    torch.cuda.synchronize()
    return event_time_ms(run, iters, stream) / iters


def _cpu_facts():
    import subprocess
    model = "unknown"
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    try:
        gcc = subprocess.run(["gcc", "-dumpfullversion"], capture_output=True,
                             text=True, timeout=10).stdout.strip()
    except (OSError, subprocess.SubprocessError):
        gcc = "?"
    flags = "?"
    with open(os.path.join(ROOT, "oracle", "Makefile")) as f:
        for line in f:
            if line.startswith("CFLAGS"):
                flags = line.split("=", 1)[1].strip()
    # the box's CPU share for one GPU is 16 threads, whatever the host has
    threads = min(16, len(os.sched_getaffinity(0)))
    return model, "gcc %s %s" % (gcc, flags), threads


def cpu_baseline(seconds=8.0):
    """The oracle (scalar C restatement) timed on this host on bounded
    samples of the same workloads: the config-2 NTT + INTT (8-limb batches,
    ~`seconds` on one thread and again on all the threads of the box's
    share), one config-4 HMult with merged rescale, and the config-3
    BConv, each on 1 thread and on all threads."""
    import numpy as np
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import _orc  # the checker library, timed here only as the CPU baseline
    from chd_primes import ntt_primes
    model, compiler, threads = _cpu_facts()
    primes = ntt_primes(30, 32)[:8]
    rng = np.random.default_rng(0xC0FFEE02)
    x = np.stack([rng.integers(0, p, N, dtype=np.uint64)
                  for p in primes]).astype(np.uint32).reshape(-1)
    pr = _orc.u32(primes)

    def ntt_rate(nthreads, budget):
        _orc.lib.orc_set_threads(nthreads)
        _orc.lib.orc_ntt_batch(x, 8, 16, pr, 0)   # warm the twiddle cache
        _orc.lib.orc_intt_batch(x, 8, 16, pr, 0)
        done, t0 = 0, time.perf_counter()
        while True:
            _orc.lib.orc_ntt_batch(x, 8, 16, pr, 0)
            _orc.lib.orc_intt_batch(x, 8, 16, pr, 0)
            done += 16
            el = time.perf_counter() - t0
            if el >= budget:
                return done / el, done, el
    one, done1, el1 = ntt_rate(1, seconds)
    many, _, _ = ntt_rate(threads, seconds / 4)

    # config 4 HMult and config 3 BConv on the oracle
    main, aux = ntt_primes(30, 24), ntt_primes(31, 8)
    r = np.random.default_rng(0xC0FFEE04)

    def uni(ps):
        return np.stack([r.integers(0, p, N, dtype=np.uint64)
                         for p in ps]).astype(np.uint32)
    b1, a1, b2, a2 = (uni(main) for _ in range(4))
    kb = np.stack([uni(main + aux) for _ in range(3)])
    ka = np.stack([uni(main + aux) for _ in range(3)])
    src_p, dst_p = ntt_primes(30, 8), ntt_primes(31, 40)
    xs = np.stack([r.integers(-((p - 1) // 2), (p - 1) // 2 + 1, N)
                   for p in src_p]).astype(np.int32)
    _, table = _orc.modswitch_consts(src_p, dst_p, 16)

    def per_call_us(fn, nthreads, reps):
        _orc.lib.orc_set_threads(nthreads)
        fn()
        t0 = time.perf_counter()
        for _ in range(reps):
            fn()
        return (time.perf_counter() - t0) / reps * 1e6
    hm = lambda: _orc.hmult(b1, a1, b2, a2, kb, ka, 24, 24, main, aux, 16, 1)  # noqa: E731
    bc = lambda: _orc.bconv(xs, table, dst_p, 16)  # noqa: E731
    hm1, hmn = per_call_us(hm, 1, 2), per_call_us(hm, threads, 4)
    bc1, bcn = per_call_us(bc, 1, 20), per_call_us(bc, threads, 40)
    _orc.lib.orc_set_threads(1)
    return {"value": one, "unit": "limb-transforms/s", "cores": 1,
            "kind": "port",
            "sample": "%d limb-transforms (8-limb NTT+INTT batches of the "
                      "config-2 primes, N=2^16) in %.1f s on 1 thread; the "
                      "same for %.1f s on %d threads; one config-4 HMult "
                      "(merged rescale) x2 / x4 and one config-3 BConv x20 / "
                      "x40" % (done1, el1, seconds / 4, threads),
            "cpu_model": model, "compiler": compiler,
            "all_cores": {"value": many, "unit": "limb-transforms/s",
                          "cores": threads},
            "hmult_us_config4": {"cores_1": hm1, "cores_%d" % threads: hmn},
            "bconv_us_config3": {"cores_1": bc1, "cores_%d" % threads: bcn}}


def run_only(chd, what, steps):
    """one workload's timed loop, for rocprofv3 runs"""
    import numpy as np
    import torch
    from chd_primes import ntt_primes
    if what == "hmult":
        return bench_hmult(chd, steps)[0] * 1e3
    if what == "hmult_cold":
        return bench_hmult(chd, steps, cold=True)[0] * 1e3
    if what == "hmult_separate":
        return bench_hmult(chd, steps, separate=True)[0] * 1e3
    if what == "hmult_levels":
        return bench_hmult_levels(chd, iters=steps)
    if what == "hrot":
        return bench_hrot(chd, steps) * 1e3
    if what == "bconv":
        return bench_bconv(chd, steps) * 1e3
    if what == "bconv_cold":
        return bench_bconv(chd, steps, cold=True) * 1e3
    if what == "hoist":
        return bench_hoist(chd, steps)[0] * 1e3
    if what == "ntt_step":
        # the headline loop (after its per-direction timings): us per step
        return bench_ntt(chd, steps, 5)[0] / steps * 1e3
    if what == "copy":
        # plain device copy of COPY_BYTES: the reference point that scales
        # the FETCH_SIZE / WRITE_SIZE counters into HBM bytes
        src = torch.ones(COPY_BYTES // 4, dtype=torch.int32, device="cuda")
        dst = torch.empty_like(src)
        stream = torch.cuda.current_stream()
        fn = lambda i: dst.copy_(src)  # noqa: E731
        fn(0)
        torch.cuda.synchronize()
        return event_time_ms(fn, steps, stream) / steps * 1e3
    # the per-direction timings of the bench line: the buffers rotate over
    # the headline's sets (more than twice the MALL), so the inputs come
    # from HBM as in the timed loop
    primes = ntt_primes(30, 32)
    plan = chd.NttPlan(primes)
    rng = np.random.default_rng(0xC0FFEE02)
    host = np.stack([np.stack([rng.integers(0, p, N, dtype=np.uint64)
                               for p in primes]) for _ in range(2)])
    base = torch.from_numpy(host.astype(np.uint32).view(np.int32)).cuda()
    nsets = ntt_sets()
    srcs = [base.clone() for _ in range(nsets)]
    dsts = [torch.empty_like(base) for _ in range(nsets)]
    stream = torch.cuda.current_stream()
    sp = ctypes.c_void_p(stream.cuda_stream)
    if what == "ntt_fwd":
        def fn(i):
            plan.forward(dsts[i % nsets], srcs[i % nsets], 32, 2, stream=sp)
    else:
        one = what == "ntt_inv_1p"

        def fn(i):
            plan.inverse(dsts[i % nsets], srcs[i % nsets], 32, 2, stream=sp,
                         single_pass=one)
    for i in range(nsets):
        fn(i)
    torch.cuda.synchronize()
    return event_time_ms(fn, steps, stream) / steps * 1e3


def traffic_from_profile():
    path = os.path.join(ROOT, "profiles", "ntt_fwd_config2_traffic.json")
    if not os.path.exists(path):
        return None
    with open(path) as f:
        return json.load(f).get("bytes_per_forward_ntt")


def main():
    args = parse()
    if args.gpus != 1:
        print("bench.py measures one GPU: the key-switch path here runs "
              "on a single MI355X and is not sharded across GPUs. Run with "
              "--gpus 1.", file=sys.stderr)
        sys.exit(2)
    import torch
    if not torch.cuda.is_available():
        print("no HIP device", file=sys.stderr)
        sys.exit(1)
    import cheddar_amd as chd

    if args.only:
        print(json.dumps({"only": args.only,
                          "us": run_only(chd, args.only, args.steps)}))
        return
    # The other workloads run first and the headline loop last: its W
    # warmup steps (0.2 ms at the driver's W = 5) do not bring an idle GPU
    # to its sustained clocks, and measured on an idle GPU the same K steps
    # read ~8 % slower.
    hoist_ms, hoist_bytes = bench_hoist(chd)
    hmult_us = bench_hmult(chd)[0] * 1e3
    hmult_cold_us, hmult_set = bench_hmult(chd, cold=True)
    hmult_cold_us *= 1e3
    hmult_sep_us = bench_hmult(chd, separate=True)[0] * 1e3
    hmult_streams_us = bench_hmult_streams(chd)
    hrot_us = bench_hrot(chd) * 1e3
    bconv_us = bench_bconv(chd) * 1e3
    bconv_cold_us = bench_bconv(chd, cold=True) * 1e3
    (ms, fwd_ms, inv_ms, warm_ms, one_ms, ok, inv1_ms, fwd2_ms,
     ms2) = bench_ntt(chd, args.steps, args.warmup)
    if not ok:
        print("NTT round trip changed the data", file=sys.stderr)
        sys.exit(1)
    lt = 128 * args.steps / (ms / 1e3)
    fwd_bytes = 64 * LIMB_TRANSFORM_BYTES
    achieved = fwd_bytes / (fwd_ms / 1e3) / 1e9
    bconv_gbs = BCONV_BYTES / (bconv_cold_us / 1e6) / 1e9
    bconv_tops = BCONV_INT8_OPS / (bconv_cold_us / 1e6) / 1e12
    hmult_gbs = HMULT_BYTES / (hmult_cold_us / 1e6) / 1e9
    hoist_gbs = hoist_bytes / (hoist_ms / 1e3) / 1e9
    line = {
        "metric": "NTT limb-transforms/s @N=2^16; HMult keyswitch us; "
                  "% HBM/MFMA roofline",
        "value": lt,
        "unit": "limb-transforms/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms / args.steps,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "u32",
        "data": "synthetic (seeded uniform residues; config-5 weights "
                "seeded N(0, 0.02), encoded by the library)",
        "config": {
            "workload": "config2: batched NTT+INTT of one ciphertext, 2 polys "
                        "x 32 limbs, N=2^16, 30-bit primes, limb-major, "
                        "buffers rotated over %d MiB, consecutive steps "
                        "over %d streams" % (0, NTT_STREAMS),
            "limb_transforms_per_step": 128,
        },
        "roofline": {
            "kernel": "forward NTT (ntt_fwd_1p: single pass, one launch, "
                      "four workgroups per limb)",
            "bound": "hbm",
            "achieved": achieved,
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": achieved / HBM_PEAK_GBS,
            "traffic": traffic_from_profile(),
        },
        "roofline_bconv": {
            "kernel": "bconv_mfma, config 3 (8 -> 40 limbs), inputs cold",
            "bound": "hbm",
            "achieved": bconv_gbs,
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": bconv_gbs / HBM_PEAK_GBS,
            "traffic": BCONV_TRAFFIC,
            "mfma": {"achieved": bconv_tops, "peak": INT8_PEAK_TOPS,
                     "unit": "TOP/s (int8, useful byte products)",
                     "frac": bconv_tops / INT8_PEAK_TOPS},
        },
        "roofline_hmult": {
            "kernel": "HMult key switch + merged rescale, config 4 (5 "
                      "launches), inputs and key cold",
            "bound": "hbm",
            "achieved": hmult_gbs,
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": hmult_gbs / HBM_PEAK_GBS,
            "traffic": HMULT_SWITCH_TRAFFIC,
            "note": "achieved = compulsory %d B (96 limbs in, 192 key limbs, "
                    "46 limbs out) / HMult time; traffic = the 5 launches' "
                    "counted HBM bytes (%d B as eight launches)"
                    % (HMULT_BYTES, HMULT_TRAFFIC),
        },
        "extra": {
            "ntt_forward_us": fwd_ms * 1e3,
            "ntt_inverse_us": inv_ms * 1e3,
            "ntt_inverse_single_pass_us": inv1_ms * 1e3,
            "ntt_forward_two_pass_us": fwd2_ms * 1e3,
            "ntt_step_us_%d_streams_two_pass_forward" % NTT_STREAMS:
                ms2 / args.steps * 1e3,
            "ntt_forward_warm_mall_us": warm_ms * 1e3,
            "ntt_step_us_one_stream": one_ms * 1e3,
            "hmult_keyswitch_us_config4": hmult_us,
            "hmult_keyswitch_us_config4_cold": hmult_cold_us,
            "hmult_then_rescale_us_config4": hmult_sep_us,
            "hrot_1234_us_config4": hrot_us,
            "hmult_us_per_op_config4_%d_streams" % NTT_STREAMS:
                hmult_streams_us,
            "bconv_us_config3_warm": bconv_us,
            "bconv_us_config3_cold": bconv_cold_us,
            "hoist_bsgs_ms_config5": hoist_ms,
            "hoist_bsgs_config5_hbm_frac": hoist_gbs / HBM_PEAK_GBS,
            "notes": "headline: the NTT+INTT loop (W warmup + K timed "
                     "steps) runs last, right after the per-direction "
                     "timings (>= 200 calls each), so it starts at "
                     "sustained clocks; right after an idle GPU the same "
                     "loop reads ~8 %% slower. Its consecutive steps "
                     "(independent ciphertexts, separate buffer sets) "
                     "alternate over %d HIP streams, so one step's loads "
                     "run beside another's butterflies; "
                     "ntt_step_us_one_stream is one step at a time on one "
                     "stream (the latency of one batch). "
                     "ntt_step_us_%d_streams_two_pass_forward: the same "
                     "loop (after the headline) with the forward on the "
                     "two-pass kernels (chd_ntt_forward_two_pass), slower "
                     "alone (ntt_forward_two_pass_us) but sharing the GPU "
                     "better with the other streams' kernels; the headline "
                     "keeps the default chd_ntt_forward. "
                     "hmult: warm = same key and inputs each step, cold = "
                     "%d MiB of distinct input/key sets rotated; host "
                     "enqueue included; hmult_then_rescale: HMult without "
                     "rescale, then a separate Rescale (warm); "
                     "hrot_1234_us_config4: HRot by 1234 slots at L=24 "
                     "(warm); "
                     "hmult_us_per_op_config4_%d_streams: "
                     "independent HMults alternating over that many "
                     "streams, one Context each, time per HMult over the "
                     "whole span (throughput, not the latency of one). "
                     "hoist: 768x768 BSGS (28 baby, 28 "
                     "giant steps, 54 rotation keys) at L=20 on the "
                     "library's encodings of a seeded N(0, 0.02) weight; "
                     "HBM fraction against the %d B of plaintexts and keys "
                     "one evaluation reads" % (NTT_STREAMS, NTT_STREAMS,
                                               hmult_set >> 20,
                                               NTT_STREAMS, hoist_bytes),
        },
    }
    line["config"]["workload"] = line["config"]["workload"].replace(
        "over 0 MiB", "over %d MiB" % (2 * ntt_sets() * 16))
    if not args.no_cpu:
        line["cpu_baseline"] = cpu_baseline()
    print(json.dumps(line))


if __name__ == "__main__":
    main()
