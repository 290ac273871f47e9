"""ctypes layouts of the kernel-level C-ABI (cheddar_kernels.h) and device
tables of a prime list, for tests that call its entries directly. Test
infrastructure only."""
import ctypes

import numpy as np

import _orc
from gpu_util import dev

P = ctypes.c_void_p
I = ctypes.c_int
LL = ctypes.c_longlong


class Tables(ctypes.Structure):
    _fields_ = [(n, P) for n in ("q", "qinv", "tw", "itw", "twist")]


class LimbMap(ctypes.Structure):
    _fields_ = [(n, I) for n in ("num_q", "skip_lo", "skip_len", "src_gap",
                                 "tab_off", "tab_gap", "cst_gap")]


class GsArgs(ctypes.Structure):
    _fields_ = [("num_bs", I), ("num_gs", I), ("add_to_dst", I),
                ("bs_b", P * 32), ("bs_a", P * 32), ("pt", (P * 32) * 8),
                ("dst_b", P * 8), ("dst_a", P * 8)]


def tables(primes, transforms=True):
    """(chd_tables of the primes, the tensors it points to); transforms:
    with the twiddles"""
    q = dev(np.array(primes, np.uint32))
    qinv = dev(np.array([pow(p, -1, 1 << 32) for p in primes], np.uint32))
    keep = [q, qinv]
    t = Tables(q=q.data_ptr(), qinv=qinv.data_ptr())
    if transforms:
        tw = [_orc.twiddles(p, 16) for p in primes]
        keep += [dev(np.stack([x[0] for x in tw])),
                 dev(np.stack([x[1] for x in tw]))]
        t.tw, t.itw = keep[2].data_ptr(), keep[3].data_ptr()
    return t, keep


def whole_map(num_q):
    """limb j is table prime j; num_q q limbs, then aux limbs"""
    return LimbMap(num_q=num_q, skip_lo=1 << 30)


def column_blocked(x):
    """limbs [..., N] in the order between a base switch's launches
    (chd_k_ntt_inv_rows): index row * 256 + col at word
    ((col >> 2) * 256 + 16 (row % 16) + row // 16) * 4 + (col & 3)"""
    out = np.empty_like(x)
    out[..., _blocked_words()] = x
    return out


def natural_order(x):
    return np.ascontiguousarray(x[..., _blocked_words()])


def _blocked_words():
    row, col = np.divmod(np.arange(1 << 16), 256)
    return ((col >> 2) * 256 + 16 * (row % 16) + row // 16) * 4 + (col & 3)


class KeyaccArgs(ctypes.Structure):
    _fields_ = ([(n, I) for n in ("num_q", "tab_off", "tab_gap", "alpha",
                                  "beta", "group_shift")] +
                [("modup", P), ("group_stride", LL), ("d", P), ("kb", P * 8),
                 ("ka", P * 8), ("key_gap", LL)] +
                [(n, P) for n in ("p_prod", "cb", "ca", "acc_b", "acc_a", "b1",
                                  "a1", "b2", "a2", "add_b", "intt_b",
                                  "intt_a")] +
                [("intt_lo", I), ("blocked", I)])


_SIGS = {
    "chd_k_ntt_inv_rows": [P, P, P, LL, P, P, LL, I, I, P],
    "chd_k_ntt_inv_cols": [P, P, P, LL, I, I, P, I, P],
    "chd_k_ntt_inv_mul": [P, P, P, LL, P, P, LL, I, I, P, I, P],
    "chd_k_ntt_fwd_groups": [P, P, P, LL, I, I, I, I, I, P],
    "chd_k_ntt_fwd_groups_batch": [P, P, P, LL, I, I, I, I, I, I, P],
    "chd_k_ntt_fwd_rows_groups": [P, P, P, P, LL, I, I, I, I, P],
    "chd_k_ntt_fwd_moddown": [P, P, P, I, P, I, I, P, P, P],
    "chd_k_ntt_fwd_moddown_multi": [P, P, P, I, I, P, LL, P, LL, I, I, P, P,
                                    P],
    "chd_k_ntt_fwd_moddown_bconv1_multi": [P, P, P, I, I, P, LL, P, P, LL, I,
                                           I, P, P, P],
    "chd_k_ntt_fwd_rows_moddown": [P, P, P, I, I, P, LL, P, LL, I, I, P, P,
                                   ctypes.c_uint32, P],
    "chd_k_modup_keyacc": [P, P, P],
}


def call(name, *args):
    """the entry with its own signature (another test may have given the
    shared function object others), tensors as their addresses, on the null
    stream; fails unless it returns 0"""
    import cheddar_amd
    fn = ctypes.CFUNCTYPE(I, *_SIGS[name])((name, cheddar_amd.lib))
    conv = [a.data_ptr() if hasattr(a, "data_ptr") else
            ctypes.addressof(a) if isinstance(a, (ctypes.Structure,
                                                  ctypes.Array)) else a
            for a in args]
    st = fn(*conv, None)
    assert st == 0, (name, cheddar_amd.lib.chd_last_error())


def pointers(ts):
    return (P * len(ts))(*[t.data_ptr() for t in ts])


def mont_mul(a, b, primes):
    """a b 2^-32 mod q, limb by limb (a, b broadcastable [limbs, N], words of
    either sign)"""
    q = np.array(primes, np.int64)[:, None]
    r = np.array([pow(1 << 32, -1, p) for p in primes], np.int64)[:, None]
    x = np.mod(a.astype(np.int64), q) * np.mod(b.astype(np.int64), q) % q
    return (x * r % q).astype(np.uint32)
