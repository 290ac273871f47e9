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
