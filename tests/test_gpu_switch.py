"""ModUp, ModDown, Rescale and the merged ModDownAndRescale against the
oracle over the shapes the column stage of a base switch distinguishes: one to
32 sources (one and two K chunks of the matrix product), destination counts
around its 16-wide tiles, more limbs than one workgroup holds (parts), and
waves whose limbs have primes on both sides of 2^30."""
import numpy as np
import pytest

import _orc
from gpu_util import N, Q30, Q31, dev, host, uniform_limbs, zeros

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def chd():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible")
    import cheddar_amd
    return cheddar_amd


def _primes(L, alpha, mixed):
    aux = Q31[:alpha]
    if not mixed:
        return Q30[:L], aux
    # 30- and 31-bit primes in turn
    high = Q31[alpha:]
    return [(Q30 if i % 2 == 0 or i // 2 >= len(high) else high)[i // 2]
            if i // 2 < len(high) else Q30[i - len(high)]
            for i in range(L)], aux


@pytest.mark.parametrize("L,alpha,mixed", [
    (2, 1, False), (3, 2, True), (5, 3, True), (9, 8, False), (17, 9, True),
    (16, 16, False), (24, 8, True), (23, 17, False), (33, 31, True)])
def test_base_switch_shapes(chd, L, alpha, mixed):
    main, aux = _primes(L, alpha, mixed)
    assert len(set(main + aux)) == L + alpha
    ctx = chd.Context(chd.Param(main, aux, [(L - 1, 0), (L, 0)]))
    r = np.random.default_rng(0x5317 + 64 * L + alpha)
    primes = main + aux
    x = uniform_limbs(r, primes)
    # the ends of the residue range, whole rows and columns of them
    q = np.array(primes, np.uint32)[:, None]
    x[:, :256] = 0
    x[:, 256:512] = q - 1
    x[:, 7::256] = q - 1
    xq = np.ascontiguousarray(x[:L])
    beta = ctx.beta(1)
    outs = [zeros(L + alpha, N) for _ in range(beta)]
    ctx.mod_up(1, outs, dev(xq))
    want = _orc.mod_up(xq, main, aux, 16)
    for g in range(beta):
        assert np.array_equal(host(outs[g]), want[g]), "group %d" % g
    out = zeros(L, N)
    ctx.mod_down(1, out, dev(x))
    assert np.array_equal(host(out), _orc.mod_down(x, primes, L, 16))
    out = zeros(L - 1, N)
    ctx.mod_down_and_rescale(1, out, dev(x))
    assert np.array_equal(host(out), _orc.mod_down(x, primes, L - 1, 16))
    ctx.rescale_poly(1, out, dev(xq))
    assert np.array_equal(host(out), _orc.mod_down(xq, main, L - 1, 16))


@pytest.mark.parametrize("wide,L", [
    (False, 17), (False, 18), (False, 25), (False, 26), (True, 23),
    (True, 24), (True, 33), (True, 34), (True, 41), (True, 42)])
def test_rescale_around_the_single_pass_limits(chd, wide, L):
    """Rescale of one polynomial and of two on both sides of the limb counts
    where the single pass and the column stage take turns: 24 and 2 x 16
    destinations below 2^30; 32, 2 x 22 and 2 x 32 to 2 x 40 with larger
    ones"""
    main = [p for pair in zip(Q30[:21], Q31[8:29]) for p in pair] if wide \
        else Q30[:26]
    main = main[:L]
    ctx = chd.Context(chd.Param(main, Q31[:8], [(L - 1, 0), (L, 0)]))
    r = np.random.default_rng(0x5E5C + 64 * wide + L)
    q = np.array(main, np.uint32)[:, None]
    x = [uniform_limbs(r, main) for _ in range(2)]
    for y in x:
        y[:, :256] = q - 1
        y[:, 256:512] = 0
        y[-1, 512:768] = q[-1] // 2 + np.arange(256) % 2  # either sign
    want = [_orc.rescale(y, main, L, 1, 16) for y in x]
    res = (zeros(L - 1, N), zeros(L - 1, N))
    ctx.rescale(1, res, (dev(x[0]), dev(x[1])))
    assert np.array_equal(host(res[0]), want[0])
    assert np.array_equal(host(res[1]), want[1])
    one = zeros(L - 1, N)
    ctx.rescale_poly(1, one, dev(x[0]))
    assert np.array_equal(host(one), want[0])


@pytest.mark.parametrize("rot", [1, 2, 255, 256, 1 << 14, N // 2 - 1])
def test_rotation_in_the_last_row_pass(chd, rot):
    """HRot, whose automorphism runs inside ModDown's last pass, for factors
    that move columns only, rows only and both, on primes on both sides of
    2^30"""
    main, aux = _primes(4, 3, True)
    ctx = chd.Context(chd.Param(main, aux, [(i, 0) for i in range(1, 5)]))
    r = np.random.default_rng(0x607 + rot)
    L = 3
    b, a = uniform_limbs(r, main[:L]), uniform_limbs(r, main[:L])
    kb, ka = (np.stack([uniform_limbs(r, main + aux) for _ in range(2)])
              for _ in range(2))
    res = (zeros(L, N), zeros(L, N))
    ctx.hrot(L - 1, res, (dev(b), dev(a)), [dev(k) for k in kb],
             [dev(k) for k in ka], rot)
    wb, wa = _orc.hrot(b, a, kb, ka, L, 4, main, aux, 16, rot)
    assert np.array_equal(host(res[0]), wb)
    assert np.array_equal(host(res[1]), wa)
