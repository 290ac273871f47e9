"""The device encoder and decoder at the sizes their passes distinguish:
message lengths around the 256-slot blocks, coefficients below a prime, up to
2^63 and beyond, small (terminal) primes, and CRT integers of every register
width. Encoding is compared with the library's host half (pinned against the
oracle on the CPU), decoding with the oracle; both bit for bit."""
import os

import numpy as np
import pytest

import _orc
import ckks_encode as E
from gpu_util import N, config4, dev, host, uniform_limbs, zeros

pytestmark = pytest.mark.gpu
PARAMS = os.path.join(os.path.dirname(__file__), "golden", "params")


@pytest.fixture(scope="module")
def chd():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible")
    import cheddar_amd
    return cheddar_amd


@pytest.fixture(scope="module")
def ctx(chd):
    main, aux, levels = config4()
    return chd.Context(chd.Param(main, aux, levels))


@pytest.fixture(scope="module")
def boot(chd):
    with open(os.path.join(PARAMS, "bootparam_35.json")) as f:
        return chd.Context(chd.Param.from_json(f.read()))


def _check_encode(c, primes, level, num_aux, scale, msg):
    dst = zeros(len(primes), N)
    slots = c.encode(level, num_aux, scale, msg, dst)
    mx, want_slots = c.param.encode_coefficients(level, num_aux, scale, msg)
    assert slots == want_slots
    want = _orc.ntt_batch(mx.reshape(-1), 16, primes, mont=1)
    assert np.array_equal(host(dst), want.reshape(len(primes), N))


@pytest.mark.parametrize("length", [1, 2, 3, 100, 255, 256, 257, 512, 513,
                                    4097, 32767])
@pytest.mark.parametrize("log_scale", [30, 55, 75])
def test_encode_lengths_and_scales(ctx, length, log_scale):
    r = np.random.default_rng(length + log_scale)
    msg = r.uniform(-1, 1, length) + 1j * r.uniform(-1, 1, length)
    msg *= 10.0 ** r.integers(-3, 4, length)
    p = ctx.param
    _check_encode(ctx, p.main[:3] + p.aux, 2, 8, 2.0 ** log_scale, msg)


@pytest.mark.parametrize("msg,scale", [
    ([0.0, -0.0, 1e-300], 1.0), ([1e300, -1e300], 1.0),
    ([1e295 + 1j, 3.0], 2.0 ** 30), ([2.0 ** 62, -(2.0 ** 63)], 1.0),
    ([2.0 ** 40] * 300, 2.0 ** 200)])
def test_encode_extreme_values(ctx, msg, scale):
    p = ctx.param
    _check_encode(ctx, p.main[:2], 1, 0, scale, np.array(msg, np.complex128))


def test_encode_small_primes(boot):
    # levels mostly of terminal primes (2^25): scaled values exceed them
    p = boot.param
    for level in (0, 3, 9):
        m, t = p.level_config[level]
        primes = p.ter[:t][::-1] + p.main[:m]
        r = np.random.default_rng(level)
        msg = r.uniform(-1, 1, 700) + 1j * r.uniform(-1, 1, 700)
        _check_encode(boot, primes, level, 0, 2.0 ** 45, msg)


def _oracle_decode(primes, pt, slots, scale):
    icrt = E.icrt_constants(primes, N)
    scaled = np.stack([
        _orc.intt_mult_const(pt[i], 16, q, icrt[i], 0).view(np.uint32)
        for i, q in enumerate(primes)])
    return E.decode_values(scaled, primes, 16, slots, scale)


def _same_bits(got, want):
    for a, b in zip((got.real, got.imag), want):
        assert np.array_equal(np.ascontiguousarray(a).view(np.uint64),
                              np.ascontiguousarray(b).view(np.uint64))


@pytest.mark.parametrize("limbs,slots", [
    (1, 1), (2, 2), (3, 256), (4, 512), (7, 128), (8, 64), (9, 1024),
    (15, 32), (17, 16), (23, 512), (24, 256)])
def test_decode_widths(ctx, limbs, slots):
    # uniform residues: values over the whole range (-Q / 2, Q / 2]
    primes = ctx.param.main[:limbs]
    x = uniform_limbs(np.random.default_rng(limbs), primes)
    x[:, :64] = 0
    got = ctx.decode(limbs - 1, 2.0 ** 30, slots, dev(x))
    want = _oracle_decode(primes, x, slots, 2.0 ** 30)
    _same_bits(got, want)


@pytest.mark.parametrize("level", [0, 12, 19, 24])
def test_decode_boot_levels(boot, level):
    p = boot.param
    m, t = p.level_config[level]
    primes = p.ter[:t][::-1] + p.main[:m]
    x = uniform_limbs(np.random.default_rng(level), primes)
    got = boot.decode(level, 2.0 ** 35, 64, dev(x))
    want = _oracle_decode(primes, x, 64, 2.0 ** 35)
    _same_bits(got, want)
