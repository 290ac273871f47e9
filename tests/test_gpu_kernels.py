"""Entries of the kernel-level C-ABI that handlers call only in chains, each
against the oracle on primes on both sides of 2^30: the passes of the inverse
transform on their own and the order of the data between them."""
import numpy as np
import pytest

import _orc
import raw_kernels as rk
from gpu_util import N, Q30, Q31, dev, host, uniform_limbs, zeros

pytestmark = pytest.mark.gpu

PRIMES = [Q30[0], Q31[0], Q30[1], Q31[30], Q30[29]]
L = len(PRIMES)


@pytest.fixture(scope="module", autouse=True)
def device():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible")


@pytest.fixture(scope="module")
def tab():
    return rk.tables(PRIMES)


def _limbs(r, primes=PRIMES):
    x = uniform_limbs(r, primes)
    x[:, :256] = np.array(primes, np.uint32)[:, None] - 1
    x[:, 256:512] = 0
    return x


def _consts(r, primes=PRIMES):
    return np.array([r.integers(1, p) for p in primes], np.uint32)


def _intt(x, cst, centre, primes=PRIMES):
    return np.stack([_orc.intt_mult_const(x[i], 16, p, int(cst[i]), centre)
                     for i, p in enumerate(primes)]).view(np.uint32)


@pytest.mark.parametrize("product", [False, True])
@pytest.mark.parametrize("centre", [0, 1])
def test_inverse_passes(tab, product, centre):
    """the column-blocked output of the inverse row pass, put back in order
    on the host and finished by the column pass, and the whole inverse of a
    product"""
    r = np.random.default_rng(0x1201 + 2 * product + centre)
    x, y, cst = _limbs(r), _limbs(r), _consts(r)
    m = rk.whole_map(L)
    dx, dy, dc = dev(x), dev(y), dev(cst)
    want = _intt(rk.mont_mul(x, y, PRIMES) if product else x, cst, centre)
    blocked = zeros(L, N)
    rk.call("chd_k_ntt_inv_rows", tab[0], m, blocked, 0, dx,
            dy if product else None, 0, L, 1)
    out = dev(rk.natural_order(host(blocked)))
    rk.call("chd_k_ntt_inv_cols", tab[0], m, out, 0, L, 1, dc, centre)
    assert np.array_equal(host(out), want)
    if product:
        out = zeros(L, N)
        rk.call("chd_k_ntt_inv_mul", tab[0], m, out, 0, dx, dy, 0, L, 1, dc,
                centre)
        assert np.array_equal(host(out), want)
