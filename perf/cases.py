"""The workloads whose speed this framework is judged by, as a user's program
runs them through the public Python binding: transforms, base conversion,
ciphertext products and rotations, plaintext products with their rescale,
hoisted linear transforms, and the encoder in both directions.

listed() gives the fixed cases, draw() one more of the same ranges. Prime
chains: "c4" is the 24 + 8 prime chain of the benchmark (30-bit main primes,
31-bit auxiliary ones, dnum 3); "boot30", "boot35" and "boot40" are the
bootstrapping parameter files (terminal primes, dnum 4), whose main primes lie
on both sides of 2^30.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "cheddar-fhe_amd", "python"))

import cheddar_amd as chd  # noqa: E402
from chd_primes import ntt_primes  # noqa: E402

N = 1 << 16
LIMB = 4 * N
SCALE = float(1 << 30)
PARAM_FILES = {"boot30": "bootparam_30.json", "boot35": "bootparam_35.json",
               "boot40": "bootparam_40.json"}


def listed():
    return [
        # one limb there and back: the smallest call, all latency (a single
        # residue polynomial of the largest word-size prime)
        {"name": "ntt_one_limb", "kind": "ntt", "bits": 31, "limbs": 1,
         "polys": 1, "mont": False, "in_place": False},
        # both polynomials of a full ciphertext there and back (the headline
        # benchmark's batch, one at a time)
        {"name": "ntt_ciphertext", "kind": "ntt", "bits": 30, "limbs": 32,
         "polys": 2, "mont": False, "in_place": False},
        # a standalone base conversion, as ModUp raises one dnum group
        {"name": "bconv_8_40", "kind": "bconv", "src": 8, "dst": 40},
        # ciphertext product with merged rescale at the top of the chain:
        # the key switch that every evaluation spends most of its time in
        {"name": "hmult_top", "kind": "hmult", "chain": "c4", "level": 23,
         "rescale": "merged"},
        # the same near the end of a computation (5 limbs, one dnum group),
        # where launches and latency count
        {"name": "hmult_low", "kind": "hmult", "chain": "c4", "level": 4,
         "rescale": "merged"},
        # product, then a separate rescale, on a bootstrapping parameter set
        # at its default encryption level: terminal primes, a shifted first
        # dnum group, restored primes
        {"name": "hmult_then_rescale_boot35", "kind": "hmult",
         "chain": "boot35", "level": 19, "rescale": "separate"},
        # slot rotation in the middle of the chain, last dnum group partial
        {"name": "hrot_mid", "kind": "hrot", "chain": "c4", "level": 16,
         "rot": 1234},
        # plaintext weight times ciphertext, then rescale (odd limb count)
        {"name": "pmult_rescale", "kind": "plain", "chain": "c4",
         "level": 12, "op": "pmult", "rescale": True},
        # one factor of a slot/coefficient transform: few giant steps
        {"name": "hoist_4x8", "kind": "hoist", "chain": "c4", "level": 12,
         "gs": 4, "bs": 8, "min_ks": False},
        # a 768 x 768 matrix times an encrypted vector (BERT projection):
        # 28 x 28 steps, 54 rotation keys, the largest call
        {"name": "hoist_768", "kind": "hoist", "chain": "c4", "level": 19,
         "gs": 28, "bs": 28, "min_ks": False},
        # a full-width message into a fresh plaintext
        {"name": "encode_full", "kind": "encode", "chain": "c4",
         "level": 23, "aux": False, "len": N // 2},
        # a result out of a plaintext near the end of the chain
        {"name": "decode_full", "kind": "decode", "chain": "c4",
         "level": 5, "slots": N // 2},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(
        rng.uniform(math.log(lo - 0.49 if lo > 1 else 0.6),
                    math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["ntt", "ntt", "bconv", "hmult", "hmult", "hrot",
                       "plain", "hoist", "encode", "decode"])
    chain = rng.choice(["c4", "c4", "c4", "boot30", "boot35", "boot40"])
    # a level of the chain, low ones as likely as high ones; the boot chains
    # up to their default encryption levels (above them only bootstrapping
    # itself computes)
    level = _log_int(rng, 1, 23 if chain == "c4" else 16)
    if kind == "ntt":
        polys = rng.choice([1, 1, 2, 3])
        return {"kind": kind, "bits": rng.choice([30, 31]),
                "limbs": _log_int(rng, 1, 40), "polys": polys,
                "mont": rng.random() < 0.5, "in_place": rng.random() < 0.5}
    if kind == "bconv":
        return {"kind": kind, "src": _log_int(rng, 1, 24),
                "dst": _log_int(rng, 1, 48)}
    if kind == "hmult":
        return {"kind": kind, "chain": chain, "level": level,
                "rescale": rng.choice(["merged", "merged", "separate",
                                       "none"])}
    if kind == "hrot":
        return {"kind": kind, "chain": chain, "level": level,
                "rot": _log_int(rng, 1, N // 2 - 1)}
    if kind == "plain":
        return {"kind": kind, "chain": chain, "level": level,
                "op": rng.choice(["pmult", "pmult", "add", "mult_const"]),
                "rescale": rng.random() < 0.6}
    if kind == "hoist":
        min_ks = rng.random() < 0.2
        top = 10 if min_ks else 27
        return {"kind": kind, "chain": "c4",
                "level": _log_int(rng, 2, 19), "gs": _log_int(rng, 1, top),
                "bs": _log_int(rng, 2, top), "min_ks": min_ks}
    if kind == "encode":
        return {"kind": kind, "chain": chain, "level": level,
                "aux": rng.random() < 0.3, "len": _log_int(rng, 1, N // 2)}
    # decoding needs the message to fit the modulus: at least two primes
    return {"kind": "decode", "chain": chain, "level": max(2, level),
            "slots": 1 << rng.randint(0, 15)}


# ------------------------------------------------------------- parameters

@functools.lru_cache(maxsize=None)
def _param(chain):
    if chain == "c4":
        p = chd.Param(ntt_primes(30, 24), ntt_primes(31, 8),
                      [(i, 0) for i in range(1, 25)])
        p.ter, p.level_config = [], [(i, 0) for i in range(1, 25)]
        return p
    with open(os.path.join(ROOT, "tests", "golden", "params",
                           PARAM_FILES[chain])) as f:
        return chd.Param.from_json(f.read())


@functools.lru_cache(maxsize=None)
def _context(chain):
    """one context per parameter set, kept for the whole program"""
    return chd.Context(_param(chain))


def _q_primes(chain, level):
    """q primes of a level in limb order: terminal ones reversed, then main"""
    p = _param(chain)
    main, ter = p.level_config[level]
    return list(reversed(p.ter[:ter])) + p.main[:main]


def _key_primes(chain):
    p = _param(chain)
    return list(reversed(p.ter)) + p.main + p.aux


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _residues(gen, primes):
    """uniform canonical residues, one limb per prime"""
    q = torch.tensor(primes, dtype=torch.int64, device="cuda")[:, None]
    x = torch.randint(0, 1 << 62, (len(primes), N), dtype=torch.int64,
                      device="cuda", generator=gen)
    return (x % q).to(torch.int32)


def _limbs(n):
    return torch.empty(n, N, dtype=torch.int32, device="cuda")


def _key(gen, chain, beta):
    primes = _key_primes(chain)
    return ([_residues(gen, primes) for _ in range(beta)],
            [_residues(gen, primes) for _ in range(beta)])


def _beta(chain):
    p = _param(chain)
    return -(-(len(p.main) + len(p.ter)) // p.alpha)


def _message(seed, n):
    r = np.random.default_rng(seed)
    return r.uniform(-1, 1, n) + 1j * r.uniform(-1, 1, n)


def _ntt_primes(case):
    # a 31-bit chain starts at the largest prime below 2^31
    return ntt_primes(case["bits"], case["limbs"])


# ----------------------------------------------------------------- the cases

def prepare(case, seed):
    kind = case["kind"]
    gen = _gen(seed)
    st = {"case": case}
    if kind == "ntt":
        primes = _ntt_primes(case)
        st["plan"] = chd.NttPlan(primes)
        st["x"] = torch.stack([_residues(gen, primes)
                               for _ in range(case["polys"])])
        st["y"] = torch.empty_like(st["x"])
        st["back"] = torch.empty_like(st["x"])
        return st
    if kind == "bconv":
        src, dst = ntt_primes(30, case["src"]), ntt_primes(31, case["dst"])
        st["plan"] = chd.BconvPlan(src, dst)
        q = torch.tensor(src, dtype=torch.int32, device="cuda")[:, None]
        x = _residues(gen, src)
        st["x"] = torch.where(x > q // 2, x - q, x)
        st["y"] = _limbs(case["dst"])
        return st
    chain, level = case["chain"], case["level"]
    ctx = st["ctx"] = _context(chain)
    primes = _q_primes(chain, level)
    if kind in ("encode", "decode"):
        limbs = len(primes)
        if kind == "encode":
            limbs += ctx.param.alpha if case["aux"] else 0
            st["msg"] = _message(seed, case["len"])
            st["y"] = _limbs(limbs)
        else:
            st["y"] = _limbs(limbs)
            ctx.encode(level, 0, SCALE, _message(seed, case["slots"]), st["y"])
        return st
    low = len(_q_primes(chain, level - 1))
    st["a"] = (_residues(gen, primes), _residues(gen, primes))
    if kind == "hmult":
        st["b"] = (_residues(gen, primes), _residues(gen, primes))
        st["key"] = _key(gen, chain, _beta(chain))
        merged = case["rescale"] == "merged"
        st["prod"] = tuple(_limbs(low if merged else len(primes))
                           for _ in range(2))
        st["res"] = tuple(_limbs(low) for _ in range(2))
    elif kind == "hrot":
        st["key"] = _key(gen, chain, _beta(chain))
        st["res"] = tuple(_limbs(len(primes)) for _ in range(2))
    elif kind == "plain":
        if case["op"] == "pmult":
            st["b"] = [_residues(gen, primes)]
        elif case["op"] == "add":
            st["b"] = [_residues(gen, primes) for _ in range(2)]
        else:
            st["cst"] = _residues(gen, primes)[:, 0].contiguous()
        st["prod"] = [_limbs(len(primes)) for _ in range(2)]
        st["res"] = tuple(_limbs(low) for _ in range(2))
    else:
        bs = list(range(case["bs"]))
        gs = [case["bs"] * k for k in range(case["gs"])]
        ext = primes + ctx.param.aux
        pts = {(g, b): _residues(gen, ext) for g in gs for b in bs}
        h = st["h"] = chd.Hoist(ctx, level, gs, bs, pts)
        st["keys"] = {r: _key(gen, chain, _beta(chain))
                      for r in h.required_rotations(case["min_ks"])}
        st["res"] = tuple(_limbs(low) for _ in range(2))
    return st


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "ntt":
        plan, x, y, back = (state[k] for k in ("plan", "x", "y", "back"))
        n, p = case["limbs"], case["polys"]
        if not case["in_place"]:
            plan.forward(y, x, n, p, mont_conv=case["mont"])
            plan.inverse(back, y, n, p, mont_conv=case["mont"])
            return y, back
        # in place: the transform replaces its input, the inverse restores it
        plan.forward(x, x, n, p, mont_conv=case["mont"])
        y.copy_(x)
        plan.inverse(x, x, n, p, mont_conv=case["mont"])
        return y, x
    if kind == "bconv":
        state["plan"].apply(state["y"], state["x"])
        return state["y"]
    ctx = state["ctx"]
    if kind == "encode":
        slots = ctx.encode(case["level"],
                           ctx.param.alpha if case["aux"] else 0, SCALE,
                           state["msg"], state["y"])
        return state["y"], slots
    if kind == "decode":
        z = ctx.decode(case["level"], SCALE, case["slots"], state["y"])
        return z.real, z.imag
    level, res = case["level"], state["res"]
    if kind == "hmult":
        kb, ka = state["key"]
        merged = case["rescale"] == "merged"
        ctx.hmult(level, state["prod"], state["a"], state["b"], kb, ka,
                  rescale=merged)
        if case["rescale"] == "separate":
            ctx.rescale(level, res, state["prod"])
            return res
        return state["prod"]
    if kind == "hrot":
        kb, ka = state["key"]
        ctx.hrot(level, res, state["a"], kb, ka, case["rot"])
        return res
    if kind == "plain":
        prod = state["prod"]
        ctx.elementwise(level, 0, case["op"], prod, list(state["a"]),
                        b=state.get("b"), cst=state.get("cst"))
        if not case["rescale"]:
            return tuple(prod)
        ctx.rescale(level, res, prod)
        return res
    state["h"].run(res, state["a"], state["keys"], min_ks=case["min_ks"])
    return res


# ----------------------------------------------------------------- the floor

# operations of one limb transform: 16 stages of N / 2 butterflies, each one
# modular product and two modular sums
_NTT_OPS = 16 * (N // 2) * 3


def _down_ops(src, dst):
    return (src + dst) * _NTT_OPS + 2 * N * src * dst


def _key_switch(num_q, alpha, beta):
    """(key bytes, operations) of ModUp and the inner product"""
    ext = num_q + alpha
    ops = ((num_q + beta * ext - num_q) * _NTT_OPS +
           2 * N * (beta * ext - num_q) * min(alpha, num_q) +
           4 * N * beta * ext)
    return 2 * beta * ext * LIMB, ops


def work(case):
    kind = case["kind"]
    if kind == "ntt":
        n = case["limbs"] * case["polys"]
        return {"bytes": 3 * n * LIMB, "flops": 2 * n * _NTT_OPS}
    if kind == "bconv":
        return {"bytes": (case["src"] + case["dst"]) * LIMB,
                "flops": 2 * N * case["src"] * case["dst"]}
    p = _param(case["chain"])
    alpha = p.alpha
    L = len(_q_primes(case["chain"], case["level"]))
    fft = 5 * (N // 2) * 15
    if kind == "encode":
        L += alpha if case["aux"] else 0
        return {"bytes": L * LIMB + 16 * case["len"],
                "flops": fft + L * _NTT_OPS}
    if kind == "decode":
        return {"bytes": L * LIMB + 16 * case["slots"],
                "flops": fft + L * _NTT_OPS + 2 * N * L * L}
    low = len(_q_primes(case["chain"], case["level"] - 1))
    off = len(p.ter) - p.level_config[case["level"]][1]
    beta = -(-(L + off) // alpha) - off // alpha
    drop = max(1, L - low)
    kb, kops = _key_switch(L, alpha, beta)
    if kind == "hmult":
        out = L if case["rescale"] == "none" else low
        return {"bytes": (4 * L + 2 * out) * LIMB + kb,
                "flops": kops + 10 * N * L + 2 * _down_ops(alpha + drop, out)}
    if kind == "hrot":
        return {"bytes": 4 * L * LIMB + kb,
                "flops": kops + 2 * _down_ops(alpha, L)}
    if kind == "plain":
        other = {"pmult": L, "add": 2 * L, "mult_const": 0}[case["op"]]
        out = low if case["rescale"] else L
        return {"bytes": (2 * L + other + 2 * out) * LIMB,
                "flops": 4 * N * L + (2 * _down_ops(drop, low)
                                      if case["rescale"] else 0)}
    gs, bs, ext = case["gs"], case["bs"], L + alpha
    nkeys = min(2, gs + bs - 2) if case["min_ks"] else gs + bs - 2
    ptl = L if case["min_ks"] else ext
    switches = gs + bs - 2
    return {"bytes": (2 * L + 2 * low + gs * bs * ptl) * LIMB + nkeys * kb,
            "flops": 4 * N * gs * bs * ptl + switches * kops +
            (gs - 1) * _down_ops(alpha, L) + 2 * _down_ops(alpha + drop, low)}


# --------------------------------------------------------------- correctness

def tolerance(case):
    # residues are whole numbers fixed by the scheme, and the decoder's
    # floating-point steps have a fixed order: every output is pinned bit
    # for bit
    return "exact"


def _root(q):
    """2N-th root of unity of the transform: g^((q - 1) / 2N) for the
    smallest generator g of Z_q"""
    factors, m, f = [], q - 1, 2
    while f * f <= m:
        if m % f == 0:
            factors.append(f)
            while m % f == 0:
                m //= f
        f += 1
    if m > 1:
        factors.append(m)
    g = next(g for g in range(2, q)
             if all(pow(g, (q - 1) // f, q) != 1 for f in factors))
    return pow(g, (q - 1) // (2 * N), q)


def _bitrev(bits):
    r = np.zeros(1, np.int64)
    for _ in range(bits):
        r = np.concatenate([2 * r, 2 * r + 1])
    return r


def _plain_ntt(x, q):
    """y[i] = sum_j x_j psi^((2 brev(i) + 1) j) mod q in 64-bit integers"""
    psi = _root(q)
    # psi^brev(j), j < N, by doubling
    w = np.ones(1, np.uint64)
    for t in range(16):
        step = np.uint64(pow(psi, N >> (t + 1), q))
        w = np.concatenate([w, w * step % np.uint64(q)])
    y = x.astype(np.uint64).reshape(1, N)
    qq = np.uint64(q)
    for _ in range(16):
        m, half = y.shape[0], y.shape[1] // 2
        b = y[:, half:] * w[m:2 * m, None] % qq
        a = y[:, :half]
        y = np.stack([(a + b) % qq, (a + qq - b) % qq], 1).reshape(2 * m, half)
    return y.reshape(N)


def exact(case, seed):
    kind = case["kind"]
    if kind == "ntt" and case["limbs"] * case["polys"] <= 64:
        primes = _ntt_primes(case)
        st = prepare(case, seed)
        x = st["x"].cpu().numpy()
        y = np.empty_like(x)
        back = x.copy()
        for p in range(case["polys"]):
            for i, q in enumerate(primes):
                v = x[p, i].astype(np.uint64)
                if case["mont"]:
                    v = v * np.uint64((1 << 32) % q) % np.uint64(q)
                y[p, i] = _plain_ntt(v, q).astype(np.int32)
                # the inverse's Montgomery conversion undoes the forward's
        return torch.from_numpy(y), torch.from_numpy(back)
    if kind == "bconv" and case["src"] * case["dst"] <= 640:
        st = prepare(case, seed)
        src, dst = ntt_primes(30, case["src"]), ntt_primes(31, case["dst"])
        x = st["x"].cpu().numpy().astype(np.int64)
        out = np.zeros((len(dst), N), np.int64)
        for k, p in enumerate(dst):
            for i, q in enumerate(src):
                # qhat_i 2^32 mod p: the conversion's result is in
                # Montgomery form
                t = pow(2, 32, p)
                for j, r in enumerate(src):
                    if j != i:
                        t = t * r % p
                out[k] = (out[k] + x[i] % p * t % p) % p
        return torch.from_numpy(out.astype(np.int32))
    if kind == "decode":
        s = case["slots"]
        n = 2 * s
        z = _message(seed, s)
        idx = np.array([pow(5, j, 4 * s) for j in range(s)], np.int64)
        zeta = np.exp(2j * np.pi * np.arange(n) / (2 * n))
        # the coefficients the encoder stores: the message's inverse
        # embedding, scaled and truncated
        full = np.zeros(n, np.complex128)
        full[(idx - 1) // 2] = z
        full[((-idx) % (2 * n) - 1) // 2] = np.conj(z)
        a = np.trunc((np.fft.fft(full) / n / zeta).real * SCALE) / SCALE
        out = (np.fft.ifft(a * zeta) * n)[(idx - 1) // 2]
        return np.ascontiguousarray(out.real), np.ascontiguousarray(out.imag)
    # the key switches, hoisted transforms and the encoder return whole
    # residues only, and a plain 64-bit restatement of them takes minutes
    return None
