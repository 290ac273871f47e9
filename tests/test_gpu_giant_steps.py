"""The plaintext accumulation of up to eight giant steps at every count it is
compiled for, with baby steps that fill its pairs and ones that do not, absent
pairs, and residues at the ends of the range, on primes on both sides of
2^30: bit-exact against the oracle's hoisted evaluation."""
import numpy as np
import pytest

import hoist_ref
from gpu_util import N, Q30, Q31, dev, host, uniform_limbs, zeros

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gs,bs,absent", [
    (1, 3, 0), (2, 1, 0), (2, 4, 1), (3, 2, 1), (4, 5, 2), (5, 3, 1),
    (8, 2, 3)])
def test_giant_step_counts(gs, bs, absent):
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible")
    import cheddar_amd
    main, aux = [Q30[0], Q31[0], Q30[1]], Q31[1:3] + Q30[2:3]
    L = len(main)
    primes = main + aux
    ctx = cheddar_amd.Context(cheddar_amd.Param(
        main, aux, [(i, 0) for i in range(1, L + 1)]))
    r = np.random.default_rng(0x6157 + 16 * gs + bs)
    bsi = list(range(bs))
    gsi = [bs * g for g in range(gs)] if bs > 1 else list(range(gs))
    pairs = [(g, b) for g in gsi for b in bsi]
    # absent pairs from the end, never a giant step's or baby step's only one
    gone = [p for p in reversed(pairs) if p[0] != gsi[0] and p[1] != 0]
    pairs = [p for p in pairs if p not in gone[:absent]]
    q = np.array(primes, np.uint32)[:, None]
    pts = {p: uniform_limbs(r, primes) for p in pairs}
    for pt in pts.values():
        pt[:, 256:768] = q - 1
    b, a = uniform_limbs(r, main), uniform_limbs(r, main)
    b[:, ::5] = q[:L] - 1
    a[:, ::7] = q[:L] - 1
    rots = sorted({x for x in bsi + gsi if x != 0})
    keys = {k: (np.stack([uniform_limbs(r, primes)]),
                np.stack([uniform_limbs(r, primes)])) for k in rots}
    if bs == 1:
        # a map of baby step 0 alone is evaluated in another order (its
        # rotations are hoisted, Hoist.cu:715-797)
        wb, wa = hoist_ref.evaluate_gs_only(
            b, a, {g: pts[(g, 0)] for g in gsi}, keys, L, L, main, aux, 16)
    else:
        wb, wa = hoist_ref.evaluate(b, a, pts, keys, L, L, main, aux, 16)
    h = cheddar_amd.Hoist(ctx, L - 1, gsi, bsi,
                          {k: dev(v) for k, v in pts.items()})
    out = (zeros(L - 1, N), zeros(L - 1, N))
    h.run(out, (dev(b), dev(a)),
          {k: ([dev(x) for x in v[0]], [dev(x) for x in v[1]])
           for k, v in keys.items()})
    assert np.array_equal(host(out[0]), wb)
    assert np.array_equal(host(out[1]), wa)


@pytest.mark.parametrize("gs,bs,add", [
    (1, 3, 0), (2, 2, 1), (3, 5, 0), (4, 4, 1), (7, 3, 0), (8, 1, 1)])
def test_signed_representatives(gs, bs, add):
    """chd_k_gs_fused takes plaintext and baby-step words in (-q, q): the
    results are the canonical words' own"""
    import ctypes
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible")
    import cheddar_amd
    import _orc
    import raw_kernels as rk
    primes = [Q30[0], Q31[0], Q30[5], Q31[7]]
    q = np.array(primes, np.int64)[:, None]
    r = np.random.default_rng(0x516E + 16 * gs + bs)

    def signed():
        """canonical words, and representatives of both signs of them"""
        x = uniform_limbs(r, primes)
        x[:, :64] = q - 1
        x[:, 64:128] = 1
        neg = r.integers(0, 2, x.shape).astype(bool)
        neg[:, :32] = False
        neg[:, 32:64] = True       # q - 1 as -1
        neg[:, 64:96] = True       # 1 as -(q - 1)
        s = np.where(neg & (x != 0), x.astype(np.int64) - q, x)
        return x, s.astype(np.int32).view(np.uint32)
    babies = [(signed(), signed()) for _ in range(bs)]
    pts = {(g, b): signed() for g in range(gs) for b in range(bs)
           if b == 0 or (g + b) % 3}
    acc = [[uniform_limbs(r, primes) if add else np.zeros((4, N), np.uint32)
            for _ in range(2)] for _ in range(gs)]
    out = [[dev(a) for a in pair] for pair in acc]
    t, keep = rk.tables(primes, transforms=False)
    a = rk.GsArgs(num_bs=bs, num_gs=gs, add_to_dst=add)
    for b, ((_, sb), (_, sa)) in enumerate(babies):
        keep += [dev(sb), dev(sa)]
        a.bs_b[b], a.bs_a[b] = (x.data_ptr() for x in keep[-2:])
    for (g, b), (_, s) in pts.items():
        keep.append(dev(s))
        a.pt[g][b] = keep[-1].data_ptr()
    for g in range(gs):
        a.dst_b[g], a.dst_a[g] = (x.data_ptr() for x in out[g])
    m = rk.whole_map(2)
    lib = cheddar_amd.lib
    lib.chd_k_gs_fused.argtypes = [rk.P, rk.P, rk.P, rk.I, rk.P]
    assert lib.chd_k_gs_fused(ctypes.byref(t), ctypes.byref(m),
                              ctypes.byref(a), 4, None) == 0
    torch.cuda.synchronize()
    for (g, b), (pt, _) in pts.items():
        for part in range(2):
            _orc.pmult_accum(acc[g][part], pt, babies[b][part][0], primes, 16)
    for g in range(gs):
        for part in range(2):
            assert np.array_equal(host(out[g][part]), acc[g][part]), (g, part)
