"""Entries of the kernel-level C-ABI that no handler calls, or calls only in
chains, each against the oracle on primes on both sides of 2^30: the passes of
the transforms on their own and the order of the data between them, the ModDown
tails in place and in a single pass, the grouped passes of ModUp, and the key
accumulation on either order of its input."""
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


def _ntt(x, primes=PRIMES):
    return _orc.ntt_batch(np.ascontiguousarray(x).reshape(-1), 16,
                          primes).reshape(len(primes), N)


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


@pytest.mark.parametrize("padded", [False, True])
@pytest.mark.parametrize("lo,hi", [(0, L), (1, 3), (0, 0)])
def test_moddown_tails(tab, lo, hi, padded):
    """NTT and ModDown epilogue of two polynomials: in place, from a source
    apart in a single pass, with a one-source conversion, and from the
    column-blocked output of the column pass with and without an
    automorphism"""
    r = np.random.default_rng(0x30D0 + 16 * lo + 2 * hi + padded)
    m = rk.whole_map(L)
    x = [_limbs(r) for _ in range(2)]
    src2 = [uniform_limbs(r, PRIMES[lo:hi]) if hi > lo
            else np.zeros((0, N), np.uint32) for _ in range(2)]
    inv, pad = _consts(r), _consts(r, PRIMES[lo:hi])
    d2 = dev(np.concatenate(src2 + [np.zeros((1, N), np.uint32)]))
    dinv, dpad = dev(inv), dev(np.append(pad, np.uint32(0)))
    dpad = dpad if padded else None

    def want(y, p):
        """of the transforms' inputs y"""
        t = -_ntt(y).astype(np.int64)
        kept = src2[p]
        if padded and hi > lo:
            kept = rk.mont_mul(kept, pad[:, None], PRIMES[lo:hi])
        t[lo:hi] += kept
        return rk.mont_mul(t, inv[:, None], PRIMES)
    stride = (hi - lo) * N
    # in place, one polynomial and both
    one = dev(x[0])
    rk.call("chd_k_ntt_fwd_moddown", tab[0], m, one, L, d2, lo, hi, dinv, dpad)
    assert np.array_equal(host(one), want(x[0], 0))
    out = [dev(v) for v in x]
    rk.call("chd_k_ntt_fwd_moddown_multi", tab[0], m, rk.pointers(out), 2, L,
            None, 0, d2, stride, lo, hi, dinv, dpad)
    for p in range(2):
        assert np.array_equal(host(out[p]), want(x[p], p)), ("in place", p)
    # single pass
    src = dev(np.concatenate(x))
    out = [zeros(L, N) for _ in range(2)]
    rk.call("chd_k_ntt_fwd_moddown_multi", tab[0], m, rk.pointers(out), 2, L,
            src, L * N, d2, stride, lo, hi, dinv, dpad)
    for p in range(2):
        assert np.array_equal(host(out[p]), want(x[p], p)), ("apart", p)
    # one centred source limb of a prime below 2^31 per polynomial
    half = (Q31[7] - 1) // 2
    s1 = r.integers(-half, half + 1, (2, N)).astype(np.int32)
    s1[:, :64], s1[:, 64:128] = half, -half
    col = _consts(r)
    out = [zeros(L, N) for _ in range(2)]
    rk.call("chd_k_ntt_fwd_moddown_bconv1_multi", tab[0], m, rk.pointers(out),
            2, L, dev(s1.view(np.uint32)), N, dev(col), d2, stride, lo, hi,
            dinv, dpad)
    for p in range(2):
        y = rk.mont_mul(np.broadcast_to(s1[p], (L, N)), col[:, None], PRIMES)
        assert np.array_equal(host(out[p]), want(y, p)), ("one source", p)
    # the row pass alone, on the column pass's output in column-blocked order
    cols = [zeros(1 + L, N) for _ in range(2)]
    for p in range(2):
        _column_pass(cols[p], x[p])
    src = dev(rk.column_blocked(np.concatenate([host(c)[1:] for c in cols])))
    for galois in (1, 5, 2 * N - 1):
        out = [zeros(L, N) for _ in range(2)]
        rk.call("chd_k_ntt_fwd_rows_moddown", tab[0], m, rk.pointers(out), 2,
                L, src, L * N, d2, stride, lo, hi, dinv, dpad, galois)
        for p in range(2):
            assert np.array_equal(host(out[p]), _orc.permute(
                want(x[p], p), 16, galois)), ("rows", galois, p)


def _column_pass(buf, x):
    """forward column pass of x (limbs of PRIMES) into buf[1:]: one group
    whose own limb 0 is left out"""
    import torch
    t, keep = rk.tables([Q30[9]] + PRIMES)
    buf[1:] = dev(x)
    m = rk.whole_map(1)
    rk.call("chd_k_ntt_fwd_groups", t, m, buf, (1 + L) * N, 1, 1, 0, 1 + L, 0)
    torch.cuda.synchronize()


# q limbs, alpha, group_shift: whole groups, a partial last one, a shifted
# first one
@pytest.mark.parametrize("num_q,alpha,shift", [(4, 2, 0), (3, 2, 0),
                                               (3, 2, 1)])
def test_grouped_passes_and_key_accumulation(num_q, alpha, shift):
    r = np.random.default_rng(0x6A0 + 16 * num_q + shift)
    primes = (PRIMES + [Q31[9]])[:num_q + alpha]
    t, keep = rk.tables(primes)
    m, total = rk.whole_map(num_q), num_q + alpha
    beta = -(-(num_q + shift) // alpha)
    own = [range(max(0, g * alpha - shift),
                 min((g + 1) * alpha - shift, num_q)) for g in range(beta)]
    gs = total * N

    def groups(n):
        return np.stack([np.stack([_limbs(r, primes) for _ in range(beta)])
                         for _ in range(n)])
    # whole transforms of two inputs, and of one
    x = groups(2)
    want = np.stack([[_ntt(x[i, g], primes) for g in range(beta)]
                     for i in range(2)])
    for g in range(beta):
        want[:, g, own[g]] = x[:, g, own[g]]
    buf = dev(x)
    rk.call("chd_k_ntt_fwd_groups_batch", t, m, buf, gs, beta, 2, alpha, shift,
            total, 1)
    assert np.array_equal(host(buf), want)
    buf = dev(x[0])
    rk.call("chd_k_ntt_fwd_groups", t, m, buf, gs, beta, alpha, shift, total,
            1)
    assert np.array_equal(host(buf), want[0])
    # column passes of both, then the row pass of one from its column-blocked
    # order
    cols = dev(x)
    rk.call("chd_k_ntt_fwd_groups_batch", t, m, cols, gs, beta, 2, alpha,
            shift, total, 0)
    blocked = dev(rk.column_blocked(host(cols)[1]))
    out = [dev(x[1, g]) for g in range(beta)]
    rk.call("chd_k_ntt_fwd_rows_groups", t, m, rk.pointers(out), blocked, gs,
            beta, alpha, shift, total)
    for g in range(beta):
        assert np.array_equal(host(out[g]), want[1, g]), g
    # key accumulation of input 1 in both orders; keys with one more q limb
    # before their aux limbs
    d, cb, ca = (_limbs(r, primes[:num_q]) for _ in range(3))
    kq = primes[:num_q] + [Q30[12]] + primes[num_q:]
    kb, ka = ([_limbs(r, kq) for _ in range(beta)] for _ in range(2))
    pp = _consts(r, primes[:num_q])
    q = np.array(primes, np.int64)[:, None]
    acc = []
    for keys, c in ((kb, cb), (ka, ca)):
        s = np.zeros((total, N), np.int64)
        s[:num_q] = rk.mont_mul(c, pp[:, None], primes[:num_q])
        for g in range(beta):
            u = want[1, g].copy()
            u[own[g]] = d[own[g]]
            s += rk.mont_mul(u, np.delete(keys[g], num_q, axis=0), primes)
        acc.append((s % q).astype(np.uint32))
    lo = num_q - 1
    cst = _consts(r, primes[lo:])
    back = [_intt(a[lo:], cst, 1, primes[lo:]) for a in acc]
    hold = [dev(v) for v in (d, cb, ca, pp)] + [dev(k) for k in kb + ka]
    for order, modup in ((0, cols[1]), (1, blocked)):
        for split in (False, True):
            ob, oa = zeros(total, N), zeros(total, N)
            ib, ia = zeros(total - lo, N), zeros(total - lo, N)
            a = rk.KeyaccArgs(num_q=num_q, alpha=alpha, beta=beta,
                              group_shift=shift, modup=modup.data_ptr(),
                              group_stride=gs, d=hold[0].data_ptr(),
                              key_gap=N, p_prod=hold[3].data_ptr(),
                              cb=hold[1].data_ptr(), ca=hold[2].data_ptr(),
                              acc_b=ob.data_ptr(), acc_a=oa.data_ptr(),
                              blocked=order)
            for g in range(beta):
                a.kb[g] = hold[4 + g].data_ptr()
                a.ka[g] = hold[4 + beta + g].data_ptr()
            if split:
                a.intt_b, a.intt_a = ib.data_ptr(), ia.data_ptr()
                a.intt_lo = lo
            rk.call("chd_k_modup_keyacc", t, a)
            end = lo if split else total
            assert np.array_equal(host(ob)[:end], acc[0][:end]), (order, split)
            assert np.array_equal(host(oa)[:end], acc[1][:end]), (order, split)
            if not split:
                continue
            mi = rk.LimbMap(num_q=total - lo, skip_lo=1 << 30, tab_off=lo)
            for got, w in ((ib, back[0]), (ia, back[1])):
                if order:
                    got = dev(rk.natural_order(host(got)))
                rk.call("chd_k_ntt_inv_cols", t, mi, got, 0, total - lo, 1,
                        dev(cst), 1)
                assert np.array_equal(host(got), w), order
