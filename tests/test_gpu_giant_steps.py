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
