"""The standalone transforms on primes on both sides of 2^30 in one call, at
limb counts around the sizes where the launch changes (tile width of the
column passes, two passes or one), on residues that include the ends of the
range: bit-exact against the CPU oracle."""
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


@pytest.mark.parametrize("limbs,polys", [
    (1, 1), (12, 1), (13, 1), (4, 4), (17, 1), (16, 2), (33, 1), (13, 5),
    (27, 3)])
def test_ntt_mixed_primes(chd, limbs, polys):
    primes = [(Q31 if i % 2 == 0 else Q30)[i // 2] for i in range(limbs)]
    plan = chd.NttPlan(primes)
    x = np.stack([uniform_limbs(np.random.default_rng(0x477 + 64 * limbs + p),
                                primes) for p in range(polys)])
    # all-largest and all-zero columns and rows, and one polynomial's last
    # limb at the largest residue throughout
    q = np.array(primes, np.uint32)[:, None]
    x[:, :, 256:512] = q - 1
    x[:, :, 512:768] = 0
    x[:, :, 5::256] = q - 1
    x[-1, -1] = primes[-1] - 1
    flat = [np.ascontiguousarray(p).reshape(-1) for p in x]
    src = dev(x)
    y = zeros(polys, limbs, N)
    for mont in (False, True):
        want = np.stack([_orc.ntt_batch(f, 16, primes, int(mont)).reshape(
            limbs, N) for f in flat])
        plan.forward(y, src, limbs, polys, mont_conv=mont)
        assert np.array_equal(host(y), want)
        plan.forward(y, src, limbs, polys, mont_conv=mont, two_pass=True)
        assert np.array_equal(host(y), want)
        z = dev(x)
        plan.forward(z, z, limbs, polys, mont_conv=mont)
        assert np.array_equal(host(z), want)
    for mont in (False, True):
        want = np.stack([_orc.intt_batch(f, 16, primes, int(mont)).reshape(
            limbs, N) for f in flat])
        plan.inverse(y, src, limbs, polys, mont_conv=mont)
        assert np.array_equal(host(y), want)
        plan.inverse(y, src, limbs, polys, mont_conv=mont, single_pass=True)
        assert np.array_equal(host(y), want)
        z = dev(x)
        plan.inverse(z, z, limbs, polys, mont_conv=mont)
        assert np.array_equal(host(z), want)


@pytest.mark.parametrize("limbs", [3, 40])
def test_ntt_signed_representatives(chd, limbs):
    """primes above 2^30 take any representative in [-q, q), to both ends of
    it, in every form of the transform"""
    primes = Q31[:limbs]
    plan = chd.NttPlan(primes)
    x = uniform_limbs(np.random.default_rng(0x519 + limbs), primes)
    q = np.array(primes, np.int64)[:, None]
    x[:, 0:512] = 0
    x[:, 512:1024] = q - 1
    low = np.arange(N) % 3 == 0
    low[256:768] = True
    y = (x.astype(np.int64) - np.where(low, q, 0)).astype(np.int32)
    assert y.min() == -max(primes)
    src, out = dev(y.view(np.uint32)), zeros(limbs, N)
    flat = np.ascontiguousarray(x).reshape(-1)
    for mont in (False, True):
        want = _orc.ntt_batch(flat, 16, primes, int(mont)).reshape(limbs, N)
        for kw in ({}, {"two_pass": True}):
            plan.forward(out, src, limbs, mont_conv=mont, **kw)
            assert np.array_equal(host(out), want), kw
        want = _orc.intt_batch(flat, 16, primes, int(mont)).reshape(limbs, N)
        for kw in ({}, {"single_pass": True}):
            plan.inverse(out, src, limbs, mont_conv=mont, **kw)
            assert np.array_equal(host(out), want), kw
