"""Timed cases of the library: what its users have it do, through the public entry points of
seal-cuda_amd/sealhip.py (and matvec.py), from one small request to the largest batches.

A case names a kind of call and its parameters:

  mulrelin   multiply + relinearize [+ rescale] of `count` ciphertext pairs at one level
  request    BFV: multiply -> relinearize -> decrypt -> batch decode of `count` pairs
  chain      CKKS: rounds of multiply -> relinearize -> rescale over pairs at uneven levels
  matvec     baby-step giant-step matrix-vector products of `count` ciphertexts (keys and
             diagonals resident)
  rotsum     CKKS: the sum of `rotations` rotations of each of `count` ciphertexts
  encrypt    encode `count` slot vectors and encrypt them with the public key
  decrypt    decrypt `count` ciphertexts and decode them to slots
  ntt        one forward and one inverse transform of `count` polynomials

Coefficient moduli are CoeffModulus::Create's: `first` bits, then `mid` bits, then a
`special` prime; BFV at N = 8192 may take the default primes instead (mid = 0).
Ciphertexts, keys and diagonals are uniform residues, which is what encryption makes of any
message; plaintexts and slots have the magnitudes of their scale.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("seal-cuda_amd"))
import matvec  # noqa: E402
import sealhip  # noqa: E402

# CoeffModulus::BFVDefault(8192)
BFV_8192 = [0x7fffffd8001, 0x7fffffc8001, 0xfffffffc001, 0xffffff6c001, 0xfffffebc001]
T_BFV = 65537
SCALE = 2.0 ** 40


def _case(name, kind, scheme, logn, L, bits, count, **more):
    first, mid, special = bits
    return dict({"name": name, "kind": kind, "scheme": scheme, "logn": logn, "L": L, "first": first, "mid": mid,
                 "special": special, "count": count}, **more)


def listed():
    return [
        # one encrypted query of a BFV service: latency of one request at the default N = 8192
        # parameters, answer decrypted and decoded
        _case("bfv_request_n13", "request", "bfv", 13, 4, (0, 0, 0), 1),
        # one CKKS product of a shallow circuit (two levels left): the smallest CKKS program step
        _case("ckks_mul_n13_l3", "mulrelin", "ckks", 13, 3, (60, 40, 60), 1, rescale=True),
        # a ragged batch of products at N = 2^14, half way down its modulus chain
        _case("ckks_mul_n14_l7_b37", "mulrelin", "ckks", 14, 7, (60, 45, 60), 37, rescale=True),
        # one product at the largest parameter set: a program that works on one ciphertext
        _case("ckks_mul_n16_l24_one", "mulrelin", "ckks", 16, 24, (60, 60, 60), 1, rescale=False),
        # the library's headline: a full batch of products at the largest parameter set
        _case("ckks_mul_n16_l24_b128", "mulrelin", "ckks", 16, 24, (60, 60, 60), 128, rescale=False),
        # the exact-integer scheme at the same size (BEHZ base conversions)
        _case("bfv_mul_n16_l24_b32", "mulrelin", "bfv", 16, 24, (60, 60, 60), 32, rescale=False),
        # a circuit's three consecutive products over ciphertexts at uneven levels
        _case("ckks_chain_n15_p64", "chain", "ckks", 15, 15, (60, 40, 60), 64, rounds=3),
        # private inference: a 1024 x 1024 layer applied to a batch of requests, CKKS
        _case("ckks_matvec_n15_b16", "matvec", "ckks", 15, 15, (60, 40, 60), 16, baby=32, giant=32),
        # private lookup: a 4096 x 4096 matrix, BFV at the default parameters
        _case("bfv_matvec_n13_b8", "matvec", "bfv", 13, 4, (0, 0, 0), 8, baby=64, giant=64),
        # slot sums (inner products, normalisations): rotate-and-add with shared decomposition
        _case("ckks_rotsum_n16_c16", "rotsum", "ckks", 16, 24, (60, 50, 60), 16, rotations=15),
        # the client's two directions at the largest parameter set
        _case("ckks_encrypt_n16_b128", "encrypt", "ckks", 16, 24, (60, 60, 60), 128),
        _case("ckks_decrypt_n16_b128", "decrypt", "ckks", 16, 24, (60, 60, 60), 128),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    cap = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["mulrelin", "mulrelin", "mulrelin", "request", "chain", "matvec", "rotsum", "encrypt",
                           "decrypt", "ntt"])
        scheme = "bfv" if kind == "request" else "ckks" if kind in ("chain", "rotsum", "ntt") else \
            rng.choice(["ckks", "ckks", "bfv"])
        logn = rng.choice([13, 14, 15, 16])
        # security bounds the modulus, so small rings have few primes
        L = rng.randint(2, {13: 4, 14: 8, 15: 15, 16: 24}[logn])
        mid = rng.choice([40, 45, 50, 55, 60])
        bits = (60, mid, 60)
        if scheme == "bfv" and logn == 13 and L == 4:
            bits = (0, 0, 0)
        count = _log(rng, 1, 128)
        more = {}
        if kind == "mulrelin":
            more = {"rescale": rng.random() < 0.5}
        elif kind == "chain":
            L = max(L, 3)
            more = {"rounds": rng.randint(1, 2)}
        elif kind == "matvec":
            more = {"baby": rng.choice([2, 4, 8, 16, 32]), "giant": rng.choice([1, 2, 4, 8, 16, 32])}
            count = _log(rng, 1, 16)
        elif kind == "rotsum":
            more = {"rotations": rng.randint(2, 15)}
            count = _log(rng, 1, 24)
        elif kind == "ntt":
            logn = rng.choice([10, 12, 13, 14, 15, 16, 17])
            L = rng.randint(1, 24)
        c = _case("", kind, scheme, logn, L, bits, count, **more)
        del c["name"]
        if _cost(c) <= cap and _state_bytes(c) <= 56e9:
            return c


# ---------------------------------------------------------------- what a pass cannot do without

def _levels(c):
    """The chain's pairs per level: a fixed spread over [rounds + 1, L], uneven counts."""
    lo = min(c["rounds"] + 1, c["L"])
    span = c["L"] - lo + 1
    got = {}
    for p in range(c["count"]):
        lv = lo + (p * 7 + p * p // 3) % span
        got[lv] = got.get(lv, 0) + 1
    return dict(sorted(got.items()))


def _ks_ops(n, logn, L):
    """Multiply-adds of one key switch: L inverse transforms, L (L + 1) forward ones, the products
    with the key, and the division by the special prime."""
    ntt = n * logn / 2
    return L * ntt + L * (L + 1) * ntt + 2 * L * (L + 1) * n + 2 * (L + 1) * ntt


def work(c):
    n, logn, L, m = 1 << c["logn"], c["logn"], c["L"], c["count"]
    ntt, limb = n * logn / 2, n * 8
    key = 2 * L * (L + 1) * limb
    kind = c["kind"]
    if kind in ("mulrelin", "request"):
        out = 2 * (L - 1 if c.get("rescale") else L)
        by = m * (4 * L + out) * limb + key
        ops = m * (4 * L * n + _ks_ops(n, logn, L))
        if c["scheme"] == "bfv":
            ops += m * (7 * (2 * L + 1) * ntt + 5 * L * (L + 1) * n)
        if c.get("rescale"):
            ops += m * 2 * L * ntt
        if kind == "request":
            by = m * (6 * L + 1) * limb + key + L * limb
            ops += m * ((2 * L + 1) * ntt + 3 * L * n)
    elif kind == "chain":
        by, ops = key, 0
        for lv, k in _levels(c).items():
            for s in range(c["rounds"]):
                a = lv - s
                by += k * (4 * a + 2 * (a - 1)) * limb
                ops += k * (4 * a * n + _ks_ops(n, logn, a) + 2 * a * ntt)
    elif kind == "matvec":
        b, g = c["baby"], c["giant"]
        by = (b * g * L + m * 4 * L) * limb + (b + g - 2) * key
        # one decomposition for the baby steps, one key switch per giant step
        ops = m * (2 * b * g * L * n + (g - 1) * _ks_ops(n, logn, L) + L * (L + 2) * ntt +
                   (b - 1) * (2 * L * (L + 1) * n + 2 * (L + 1) * ntt))
        if c["scheme"] == "bfv":
            ops += m * 2 * (b + g) * L * ntt
    elif kind == "rotsum":
        r = c["rotations"]
        by = m * 4 * L * limb + r * key
        ops = m * (L * (L + 2) * ntt + r * 2 * L * (L + 1) * n + 2 * (L + 1) * ntt)
    elif kind == "encrypt":
        slots = n * 8
        by = m * (slots + 2 * L * limb) + 2 * (L + 1) * limb
        ops = m * ((L + 1 + 2 + 2 * L + L) * ntt + 2 * (L + 1) * n + 2 * n * logn)
    elif kind == "decrypt":
        by = m * (2 * L * limb + (L * limb if c["scheme"] == "ckks" else limb) + n * 8) + L * limb
        ops = m * (2 * L * n + L * ntt + L * n + 2 * n * logn)
    else:
        by = 2 * 2 * m * L * limb
        ops = 2 * m * L * ntt
    return {"bytes": float(by), "flops": 2.0 * ops}


def _cost(c):
    w = work(c)
    return max(w["bytes"] / 4e12, w["flops"] / 2.2e12)


def _state_bytes(c):
    n, L, m = 1 << c["logn"], c["L"], c["count"]
    limb = n * 8
    ks = m * (L * (L + 1) + 5 * L + 2)
    keys = 2 * L * (L + 1)
    extra = {"matvec": (c.get("baby", 0) + c.get("giant", 0)) * (m * 2 * L + 2 * keys) +
             c.get("baby", 0) * c.get("giant", 0) * L, "rotsum": 2 * c.get("rotations", 0) * keys,
             "chain": m * 30 * L, "encrypt": m * 8 * L, "decrypt": m * 6 * L}.get(c["kind"], 0)
    return limb * (ks + keys + extra + m * 20 * L)


# ---------------------------------------------------------------- inputs

def _moduli(c):
    n = 1 << c["logn"]
    if c["mid"] == 0:
        return list(BFV_8192)
    return sealhip.coeff_modulus_create(n, [c["first"]] + [c["mid"]] * (c["L"] - 1) + [c["special"]])


class State:
    pass


def _empty(*shape):
    return torch.empty(shape, dtype=torch.int64, device="cuda")


def _words(nbytes):
    return _empty((max(nbytes, 8) + 7) // 8)


def _uniform(t, moduli, dim, gen):
    """Uniform residues of moduli[i] at index i of dimension `dim`."""
    for i, q in enumerate(moduli):
        s = t.select(dim, i)
        s.copy_(torch.randint(0, q, s.shape, generator=gen, device="cuda", dtype=torch.int64))
    return t


def _key(s, gen):
    K = len(s.moduli)
    return _uniform(_empty(K - 1, 2, K, s.n), s.moduli, 2, gen)


def _cts(s, count, level, gen):
    return _uniform(_empty(count, 2, level, s.n), s.moduli[:level], 2, gen)


def prepare(case, seed):
    sealhip.init(0)
    s = State()
    s.case = case
    s.n = n = 1 << case["logn"]
    s.L, s.count, s.kind = case["L"], case["count"], case["kind"]
    L, m = s.L, s.count
    s.bfv = case["scheme"] == "bfv"
    s.moduli = _moduli(case)
    s.ctx = ctx = sealhip.Context(sealhip.SCHEME_BFV if s.bfv else sealhip.SCHEME_CKKS, n, s.moduli,
                                  T_BFV if s.bfv else 0)
    st = torch.cuda.current_stream().cuda_stream
    gen = torch.Generator(device="cuda").manual_seed(1000003 * (seed + 1) + 17)
    if s.kind in ("mulrelin", "request"):
        s.a, s.b, s.key = _cts(s, m, L, gen), _cts(s, m, L, gen), _key(s, gen)
        s.prod = _empty(m, 3, L, n)
        s.mw, s.kw = ctx.multiply_workspace_size(m, L), ctx.keyswitch_workspace_size(m, L)
        s.ws = _words(max(s.mw, s.kw))
        if case.get("rescale"):
            s.rw = ctx.rescale_workspace_size(m, 2, L)
            s.rs, s.out = _words(s.rw), _empty(m, 2, L - 1, n)
        if s.kind == "request":
            s.sk = _secret(s, seed, st)
            s.dw = ctx.decrypt_many_workspace_size(L, m)
            s.db, s.plain, s.slots, s.scratch = _words(s.dw), _empty(m, n), _empty(m, n), _empty(m, n)
    elif s.kind == "chain":
        s.key = _key(s, gen)
        s.groups = []
        for lv, k in _levels(case).items():
            r = range(case["rounds"])
            s.groups.append((lv, k, _cts(s, k, lv, gen), [_cts(s, k, lv - i, gen) for i in r],
                             [_empty(k, 3, lv - i, n) for i in r], [_empty(k, 2, lv - i - 1, n) for i in r]))
        s.gw = 0
        for i in range(case["rounds"]):
            pr = [(p[i].data_ptr(), k, lv - i) for lv, k, _, _, p, _ in s.groups]
            s.gw = max(s.gw, ctx.relinearize_groups_workspace_size(pr), ctx.rescale_groups_workspace_size(pr))
        s.ws = _words(s.gw)
    elif s.kind == "matvec":
        b, g = case["baby"], case["giant"]
        s.plains = _uniform(_empty(g, b, L, n), s.moduli[:L], 2, gen)
        s.baby = [_key(s, gen) for _ in range(1, b)]
        s.giant = [_key(s, gen) for _ in range(1, g)]
        s.hoisted = _hoist(s, s.baby, [ctx.galois_elt_from_step(j) for j in range(1, b)], st)
        s.mv = matvec.BsgsMatvec(ctx, n, L, b, g, s.plains.data_ptr(), [k.data_ptr() for k in s.baby],
                                 [h.data_ptr() for h in s.hoisted], [k.data_ptr() for k in s.giant], bfv=s.bfv)
        s.x = _cts(s, m, L, gen)
        s.out = torch.empty_like(s.x)
        s.rot, s.inner = _empty(b, m, 2, L, n), _empty(g, m, 2, L, n)
        s.kw = s.mv.workspace_sizes(m)
        s.ws = _words(s.kw)
    elif s.kind == "rotsum":
        s.elts = [ctx.galois_elt_from_step(1 << k if (1 << k) < n // 2 else 3) for k in range(case["rotations"])]
        s.keys = [_key(s, gen) for _ in s.elts]
        s.hoisted = _hoist(s, s.keys, s.elts, st)
        s.x = _cts(s, m, L, gen)
        s.out = torch.empty_like(s.x)
        s.kw = ctx.rotate_sum_workspace_size(m, L)
        s.ws = _words(s.kw)
    elif s.kind == "encrypt":
        # keys and encryptions draw from ChaCha20 under a 256-bit key, as the C++ API has it
        ctx.set_sampler_key(np.random.default_rng(seed).bytes(32))
        sk = _secret(s, seed, st)
        s.pk = _empty(2, len(s.moduli), n)
        ctx.keygen_public(sk.data_ptr(), 2 * seed + 2, s.pk.data_ptr(), st)
        if s.bfv:
            s.values = torch.randint(0, T_BFV, (m, n), generator=gen, device="cuda", dtype=torch.int64)
            s.plain = _empty(m, n)
        else:
            s.values = torch.rand((m, n), dtype=torch.float64, device="cuda", generator=gen) * 2 - 1
            s.plain = _empty(m, L, n)
            s.cw = ctx.ckks_encode_many_workspace_size(m)
            s.cb, s.status = _words(s.cw), torch.zeros((m,), dtype=torch.int32, device="cuda")
        s.ew = ctx.encrypt_many_workspace_size(L, m)
        s.eb, s.out, s.seed = _words(s.ew), _empty(m, 2, L, n), 7919 * seed + 5
    elif s.kind == "decrypt":
        s.sk = _secret(s, seed, st)
        s.x = _cts(s, m, L, gen)
        s.slots = _empty(m, n) if s.bfv else torch.empty((m, n), dtype=torch.float64, device="cuda")
        s.dw = ctx.decrypt_many_workspace_size(L, m)
        s.db = _words(s.dw)
        if s.bfv:
            s.plain, s.scratch = _empty(m, n), _empty(m, n)
        else:
            s.plain = _empty(m, L, n)
            s.cw = ctx.ckks_decode_many_workspace_size(L, m)
            s.cb = _words(s.cw)
            # ciphertexts of messages: c0 = NTT(message) - c1 s, with c1 uniform
            msg = torch.from_numpy(_message(case, seed)).cuda()
            s.x[:, 0].zero_()
            cs, pt = _empty(m, L, n), _empty(m, L, n)
            ctx.decrypt_many(s.x.data_ptr(), 2, m, s.sk.data_ptr(), L, cs.data_ptr(), s.db.data_ptr(), s.dw, st)
            for i, q in enumerate(s.moduli[:L]):
                pt[:, i] = torch.remainder(msg, q)
            ctx.ntt_forward(pt.data_ptr(), m, L, st)
            ctx.sub(pt.data_ptr(), cs.data_ptr(), pt.data_ptr(), m, L, st)
            s.x[:, 0] = pt
    else:
        s.fwd = _uniform(_empty(m, L, n), s.moduli[:L], 1, gen)
        s.inv = _uniform(_empty(m, L, n), s.moduli[:L], 1, gen)
    torch.cuda.current_stream().synchronize()
    return s


def _secret(s, seed, st):
    sk = _empty(len(s.moduli), s.n)
    s.ctx.keygen_secret(2 * seed + 1, sk.data_ptr(), st)
    return sk


def _hoist(s, keys, elts, st):
    hb, hw = s.ctx.hoisted_key_size(s.L), s.ctx.hoisted_key_workspace_size(s.L)
    ws, got = _words(hw), []
    for k, e in zip(keys, elts):
        got.append(_words(hb))
        s.ctx.hoisted_key_prepare(k.data_ptr(), e, s.L, got[-1].data_ptr(), ws.data_ptr(), hw, st)
    return got


def _message(case, seed):
    """Plaintext coefficients of slots in [-1, 1] at scale 2^40: about 2^40 / sqrt(N) each."""
    n, rng = 1 << case["logn"], np.random.default_rng(seed + 31)
    return np.rint(rng.standard_normal((case["count"], n)) * (SCALE / math.sqrt(n))).astype(np.int64)


# ---------------------------------------------------------------- one pass

def run(s):
    ctx, L, m, n = s.ctx, s.L, s.count, s.n
    st = torch.cuda.current_stream().cuda_stream
    if s.kind in ("mulrelin", "request"):
        ctx.multiply(s.a.data_ptr(), s.b.data_ptr(), s.prod.data_ptr(), m, L, s.ws.data_ptr(), s.mw, st)
        ctx.relinearize(s.prod.data_ptr(), s.key.data_ptr(), m, L, s.ws.data_ptr(), s.kw, st)
        if s.kind == "mulrelin" and not s.case.get("rescale"):
            return s.prod[:, :2]
        rel = s.prod[:, :2].contiguous()  # the size-2 results, packed
        if s.kind == "mulrelin":
            ctx.rescale_to_next(rel.data_ptr(), s.out.data_ptr(), m, 2, L, s.rs.data_ptr(), s.rw, st)
            return s.out
        ctx.decrypt_many(rel.data_ptr(), 2, m, s.sk.data_ptr(), L, s.plain.data_ptr(), s.db.data_ptr(), s.dw, st)
        ctx.batch_decode_many(s.plain.data_ptr(), m, s.slots.data_ptr(), s.scratch.data_ptr(), st)
        return [rel, s.slots]
    if s.kind == "chain":
        for i in range(s.case["rounds"]):
            a = [((x if i == 0 else acc[i - 1]).data_ptr(), k, lv - i) for lv, k, x, _, _, acc in s.groups]
            b = [(y[i].data_ptr(), k, lv - i) for lv, k, _, y, _, _ in s.groups]
            pr = [(p[i].data_ptr(), k, lv - i) for lv, k, _, _, p, _ in s.groups]
            out = [(acc[i].data_ptr(), k, lv - i - 1) for lv, k, _, _, _, acc in s.groups]
            ctx.ckks_multiply_groups(a, b, pr, st)
            ctx.relinearize_groups(pr, s.key.data_ptr(), s.ws.data_ptr(), s.gw, st)
            ctx.rescale_to_next_groups(pr, 3, out, s.ws.data_ptr(), s.gw, st)
        return [acc[-1] for *_, acc in s.groups]
    if s.kind == "matvec":
        s.mv.run(s.x.data_ptr(), m, s.out.data_ptr(), s.rot.data_ptr(), s.inner.data_ptr(), s.ws.data_ptr(), s.kw, st)
        return s.out
    if s.kind == "rotsum":
        ctx.rotate_sum(s.x.data_ptr(), m, L, s.elts, [h.data_ptr() for h in s.hoisted],
                       [k.data_ptr() for k in s.keys], s.out.data_ptr(), s.ws.data_ptr(), s.kw, st)
        return s.out
    if s.kind == "encrypt":
        if s.bfv:
            ctx.batch_encode_many(s.values.data_ptr(), n, n, m, s.plain.data_ptr(), st)
        else:
            ctx.ckks_encode_many(s.values.data_ptr(), n // 2, n, m, SCALE, L, s.plain.data_ptr(), s.status.data_ptr(),
                                 s.cb.data_ptr(), s.cw, st)
        ctx.encrypt_many(s.pk.data_ptr(), s.plain.data_ptr(), m, L, s.seed, s.out.data_ptr(), s.eb.data_ptr(), s.ew,
                         st)
        return s.out
    if s.kind == "decrypt":
        ctx.decrypt_many(s.x.data_ptr(), 2, m, s.sk.data_ptr(), L, s.plain.data_ptr(), s.db.data_ptr(), s.dw, st)
        if s.bfv:
            ctx.batch_decode_many(s.plain.data_ptr(), m, s.slots.data_ptr(), s.scratch.data_ptr(), st)
        else:
            ctx.ckks_decode_many(s.plain.data_ptr(), L, m, SCALE, s.slots.data_ptr(), s.cb.data_ptr(), s.cw, st)
        return [s.plain, s.slots]
    ctx.ntt_forward(s.fwd.data_ptr(), m, L, st)
    ctx.ntt_inverse(s.inv.data_ptr(), m, L, st)
    return [s.fwd, s.inv]


def tolerance(c):
    """Whole words are exact; decoded slots carry the rounding of a 64-bit FFT of N points."""
    if c["kind"] == "decrypt" and c["scheme"] == "ckks":
        return {"rel": 4e-15, "max": 4e-14}
    return "exact"


def exact(c, seed):
    """The decoded slots: the message polynomial at the odd powers zeta^(3^i) of the 2N-th root of
    unity, over the scale.  The other outputs are whole words."""
    if c["kind"] != "decrypt" or c["scheme"] != "ckks":
        return None
    n = 1 << c["logn"]
    msg = _message(c, seed).astype(np.longdouble) / np.longdouble(SCALE)
    k = np.arange(n)
    zeta = np.exp(1j * np.pi * k / n)
    at = np.empty(n // 2, dtype=np.int64)
    p = 1
    for i in range(n // 2):
        at[i] = (p - 1) // 2
        p = p * 3 % (2 * n)
    ev = np.fft.ifft(msg.astype(np.float64) * zeta, axis=1) * n
    got = ev[:, at]
    return [None, np.stack([got.real, got.imag], axis=2).reshape(c["count"], n)]
