"""Hoisted rotations on the GPU (sums and separate outputs).

shc_rotate_sum and shc_rotate_many (one ModUp of c1 for every rotation, keys prepared with
the sign-pattern correction) must give the words of summing (or listing) separate rotations -- the oracle's
applyGaloisInplace restatement, itself pinned against the reference -- for CKKS (NTT
form) and BFV (coefficient form), for positive, negative and conjugation elements, and
when c1 has zero digits (fixed on the device), is entirely zero, or has many zeros; and a
captured HIP graph of the call replays to the same words.  shc_rotate_accumulate likewise
must give the words of separate rotations summed, in every workspace that holds one.
"""
import numpy as np
import torch
import pytest

import checkers as ck
from gpu_util import empty_dev, from_dev, hip, stream, to_dev

pytestmark = pytest.mark.gpu
BFV, CKKS = 1, 2


def ws(nbytes):
    return empty_dev((max(nbytes, 8) + 7) // 8)


def run_case(scheme, logn, bits, L, count, steps, zero_digits=False, seed=0):
    """zero_digits: False; True (two zeroed coefficients of ciphertext 0's c1); or
    "heavy" (ciphertext 0's c1 entirely zero, every 16th coefficient of ciphertext 1's c1
    zero)."""
    n = 1 << logn
    moduli = ck.coeff_modulus_create(n, bits)
    K = len(moduli)
    ctx = hip().Context(scheme, n, moduli, 65537 if scheme == BFV else 0)
    rng = np.random.default_rng(seed)
    cts = ck.uniform_residues(rng, (count, 2, L, n), moduli[:L])
    if zero_digits == "heavy":
        cts[0, 1] = 0
        c1 = cts[1, 1]
        if scheme == CKKS:
            c1 = ck.ntt_rns(c1, moduli[:L], logn, inverse=True)
        c1[:, ::16] = 0
        cts[1, 1] = ck.ntt_rns(c1, moduli[:L], logn) if scheme == CKKS else c1
    elif zero_digits:
        # zero some coefficient-form digits of c1 (CKKS holds c1 in NTT form)
        c1 = cts[0, 1]
        if scheme == CKKS:
            c1 = ck.ntt_rns(c1, moduli[:L], logn, inverse=True)
        c1[:, 5] = 0
        c1[1, 17] = 0
        cts[0, 1] = ck.ntt_rns(c1, moduli[:L], logn) if scheme == CKKS else c1
    elts = [ck.galois_elt(logn, s) for s in steps]
    keys = [ck.random_key(rng, moduli, logn) for _ in steps]
    dkeys = [to_dev(k) for k in keys]
    hb = ctx.hoisted_key_size(L)
    hw = ctx.hoisted_key_workspace_size(L)
    hws = ws(hw)
    hkeys = []
    for e, dk in zip(elts, dkeys):
        h = empty_dev(((hb + 7) // 8,))
        ctx.hoisted_key_prepare(dk.data_ptr(), e, L, h.data_ptr(), hws.data_ptr(), hw, stream())
        hkeys.append(h)
    din = to_dev(cts)
    out = empty_dev((count, 2, L, n))
    many = empty_dev((len(elts), count, 2, L, n))
    rw = ctx.rotate_sum_workspace_size(count, L)
    rws = ws(rw)
    hp, kp = [h.data_ptr() for h in hkeys], [k.data_ptr() for k in dkeys]
    ctx.rotate_sum(din.data_ptr(), count, L, elts, hp, kp, out.data_ptr(), rws.data_ptr(), rw, stream())
    ctx.rotate_many(din.data_ptr(), count, L, elts, hp, kp, many.data_ptr(), rws.data_ptr(), rw, stream())
    got, got_many = from_dev(out), from_dev(many)
    for c in range(count):
        want = None
        for r, (e, k) in enumerate(zip(elts, keys)):
            rot = ck.apply_galois_keyswitch(scheme, cts[c], e, k, moduli, L, logn)
            np.testing.assert_array_equal(got_many[r, c], rot, err_msg=f"rotation {r} of ciphertext {c}")
            want = rot if want is None else ck.mod_add(want, rot, moduli)
        np.testing.assert_array_equal(got[c], want, err_msg=f"ciphertext {c}")
    # the input is untouched
    np.testing.assert_array_equal(from_dev(din), cts)


@pytest.mark.parametrize("scheme,logn,bits,L,count,steps", [
    (CKKS, 10, [60, 40, 40, 60], 3, 2, [1, 2, -1]),
    (CKKS, 13, [60, 40, 40, 40, 60], 4, 3, [1, 4, -3, 0]),
    (BFV, 12, [40, 40, 50], 2, 2, [1, -2, 0]),
    (BFV, 13, [43, 43, 44, 44, 44], 4, 1, [3, 7]),
    (CKKS, 15, [60] + [40] * 6 + [60], 5, 2, [1, 2, 4, 8]),   # a level below the first
])
def test_rotate_sum_equals_separate_rotations(scheme, logn, bits, L, count, steps):
    run_case(scheme, logn, bits, L, count, steps, seed=logn + L)


@pytest.mark.parametrize("scheme", [CKKS, BFV])
def test_rotate_sum_zero_digits_exact(scheme):
    """A zero digit at a negated position has the reference digit 0: the device lists the
    zeros and puts the products right, so the words still equal separate rotations."""
    run_case(scheme, 12, [40, 40, 50], 2, 2, [1, 2], zero_digits=True, seed=5)


@pytest.mark.parametrize("scheme", [CKKS, BFV])
def test_rotate_sum_many_zero_digits_and_zero_c1(scheme):
    run_case(scheme, 12, [40, 40, 50], 2, 2, [1, 2, -1, 3, 5], zero_digits="heavy", seed=6)


@pytest.mark.parametrize("scheme,bits,L,count,rotations", [
    # N >= 2^13: passes of up to 4 rotations share their launches, a block's waves share
    # positions from 3 ciphertexts up, one summed ModDown takes up to 15 rotations
    (CKKS, [60, 40, 50], 2, 1, 1),
    (CKKS, [60, 40, 50], 2, 9, 5),
    (CKKS, [50, 45], 1, 4, 16),
    (CKKS, [60, 55, 60], 2, 3, 17),
    (BFV, [43, 44, 44], 2, 5, 16),
    (BFV, [60, 60, 60], 2, 2, 3),
])
def test_rotation_passes(scheme, bits, L, count, rotations):
    run_case(scheme, 13, bits, L, count, list(range(1, rotations + 1)), seed=rotations)


@pytest.mark.parametrize("scheme", [CKKS, BFV])
@pytest.mark.parametrize("zeros", [True, "heavy"])
def test_rotation_passes_zero_digits(scheme, zeros):
    run_case(scheme, 13, [60, 40, 50], 2, 2, [1, 2, -1, 3, 5], zero_digits=zeros, seed=8)


@pytest.mark.parametrize("scheme,logn,bits,L,count,steps", [
    (CKKS, 12, [60, 40, 40, 60], 3, 2, [None, 1, -2]),                  # one at a time
    (CKKS, 11, [60, 40, 60], 2, 3, [1, None, 2, None]),
    (BFV, 12, [40, 40, 50], 2, 2, [0, 1, None]),
    (BFV, 10, [40, 50], 1, 1, [None, 3]),
    (CKKS, 13, [60, 40, 50, 60], 3, 3, [None] + list(range(1, 18))),    # two summed ModDowns
    (BFV, 13, [43, 44, 44], 2, 5, [1, 2, None, 3, 0, 4, 5]),            # batches around the identity
    (BFV, 14, [60, 50, 60], 2, 1, [None]),
    (CKKS, 15, [60, 40, 50, 60], 3, 5, [None, 2, 4, 6, 8, 10]),         # the fused key products
    (CKKS, 15, [60, 60], 1, 1, [3]),
    (BFV, 15, [60, 50, 60], 2, 2, [1, 0]),
    (CKKS, 16, [60, 40, 60], 2, 3, [None, 1, 2, 3]),
    (BFV, 16, [60, 60], 1, 1, [1, None]),
    (CKKS, 17, [60, 50, 60], 2, 1, [1, 2, None, 3, 4, 5]),              # several keys, unfused
    (BFV, 17, [60, 60], 1, 2, [2, 1]),
])
def test_rotate_accumulate(scheme, logn, bits, L, count, steps):
    accumulate_case(scheme, logn, bits, L, count, steps)


@pytest.mark.parametrize("scheme,logn,bits,count", [
    (CKKS, 13, [60, 40, 60], 3), (BFV, 13, [43, 44, 44], 2), (CKKS, 15, [60, 40, 60], 2), (BFV, 17, [60, 60, 60], 1)])
def test_rotate_accumulate_in_smaller_workspaces(scheme, logn, bits, count):
    """Every workspace from one rotation's need up gives the words, with as many rotations at a
    time as it holds (regions of whole limbs: digits, T, products, sums, corrections)."""
    L, n = 2, 1 << logn
    for nb in (1, 2, 3):
        T = 6 * (1 if logn in (15, 16) else nb)
        accumulate_case(scheme, logn, bits, L, count, [1, 2, None, 3, 4, 5],
                        (T + nb * (3 * L + 2) + 4 * L + 2) * count * n * 8, refused=nb == 1)


@pytest.mark.parametrize("scheme,logn,count", [(CKKS, 13, 1040), (BFV, 13, 1040), (CKKS, 15, 264)])
def test_rotation_launch_forms_agree(scheme, logn, count):
    """Batches whose permuted inverse transforms and permuted ModDowns pass 2^26 words (16 values
    per thread) against the same ciphertexts in slices below (4 values), which the oracle
    checks above."""
    L, n = 2, 1 << logn
    moduli = ck.coeff_modulus_create(n, [60, 40, 60])
    ctx = hip().Context(scheme, n, moduli, 65537 if scheme == BFV else 0)
    gen = torch.Generator(device="cuda").manual_seed(logn)
    x = torch.empty((4, count, 2, L, n), dtype=torch.int64, device="cuda")
    for i in range(L):
        x[..., i, :] = torch.randint(0, moduli[i], (4, count, 2, n), generator=gen, device="cuda", dtype=torch.int64)
    rng = np.random.default_rng(logn)
    elts = [ck.galois_elt(logn, s) for s in (1, 2, -1, 3)]
    keys = [to_dev(ck.random_key(rng, moduli, logn)) for _ in elts]
    hb, hw = ctx.hoisted_key_size(L), ctx.hoisted_key_workspace_size(L)
    hws, hoisted = ws(hw), []
    for e, k in zip(elts, keys):
        hoisted.append(empty_dev(((hb + 7) // 8,)))
        ctx.hoisted_key_prepare(k.data_ptr(), e, L, hoisted[-1].data_ptr(), hws.data_ptr(), hw, stream())
    kp, hp = [k.data_ptr() for k in keys], [h.data_ptr() for h in hoisted]

    def run(x):
        m = x.shape[1]
        # room for four rotations at a time in both
        wb = max(ctx.rotate_sum_workspace_size(m, L), (24 + 4 * (3 * L + 2) + 4 * L + 2) * m * n * 8)
        buf = ws(wb)
        many, one, acc = empty_dev((4, m, 2, L, n)), empty_dev((m, 2, L, n)), empty_dev((m, 2, L, n))
        ctx.rotate_many(x.data_ptr(), m, L, elts, hp, kp, many.data_ptr(), buf.data_ptr(), wb, stream())
        ctx.rotate_sum(x.data_ptr(), m, L, elts, hp, kp, one.data_ptr(), buf.data_ptr(), wb, stream())
        ctx.rotate_accumulate(x.data_ptr(), m, L, elts, kp, acc.data_ptr(), buf.data_ptr(), wb, stream())
        torch.cuda.synchronize()
        return many, one, acc

    assert 4 * 2 * count * n > 1 << 26       # the special limbs of a pass
    assert 4 * count * L * n > 1 << 26       # the digits of a batch
    many, one, acc = run(x)
    step = count // 8 + 1
    for c in range(0, count, step):
        sl = slice(c, min(c + step, count))
        m, o, a = run(x[:, sl].contiguous())
        assert torch.equal(many[:, sl], m) and torch.equal(one[sl], o) and torch.equal(acc[sl], a)


def test_rotate_accumulate_rejects():
    logn, n, L, count = 13, 1 << 13, 2, 2
    moduli = ck.coeff_modulus_create(n, [60, 40, 60])
    ctx = hip().Context(CKKS, n, moduli)
    rng = np.random.default_rng(4)
    din = to_dev(ck.uniform_residues(rng, (3, count, 2, L, n), moduli[:L]))
    key = to_dev(ck.random_key(rng, moduli, logn))
    out = empty_dev((count, 2, L, n))
    wb = ctx.rotate_accumulate_workspace_size(count, L)
    buf = ws(wb)
    e = ck.galois_elt(logn, 1)

    def call(elts, keys, dst, w=wb):
        ctx.rotate_accumulate(din.data_ptr(), count, L, elts, keys, dst.data_ptr(), buf.data_ptr(), w, stream())

    k = key.data_ptr()
    for elts, keys, dst in (([1, e, 2], [None, k, k], out), ([1, e, 2 * n + 1], [None, k, k], out),  # no such element
                            ([1, e, e], [None, k, None], out),                                       # no key
                            ([1, e, e], [None, k, k], din[0]), ([1, e, e], [None, k, k], din[2])):   # over the input
        with pytest.raises(hip().SealHipError):
            call(elts, keys, dst)
    with pytest.raises(hip().SealHipError):
        call([e], [k], out, 0)
    call([1, e, e], [None, k, k], out)


def accumulate_case(scheme, logn, bits, L, count, steps, ws_bytes=None, refused=False):
    """ws_bytes: None for the size that is asked for.  refused: one byte less is too small."""
    n = 1 << logn
    moduli = ck.coeff_modulus_create(n, bits)
    ctx = hip().Context(scheme, n, moduli, 65537 if scheme == BFV else 0)
    rng = np.random.default_rng(len(steps) + logn)
    cts = ck.uniform_residues(rng, (len(steps), count, 2, L, n), moduli[:L])
    elts = [1 if s is None else ck.galois_elt(logn, s) for s in steps]
    keys = [None if s is None else ck.random_key(rng, moduli, logn) for s in steps]
    dkeys = [None if k is None else to_dev(k) for k in keys]
    din, out = to_dev(cts), empty_dev((count, 2, L, n))
    wb = ctx.rotate_accumulate_workspace_size(count, L) if ws_bytes is None else ws_bytes
    buf = ws(wb)
    args = (din.data_ptr(), count, L, elts, [None if k is None else k.data_ptr() for k in dkeys], out.data_ptr(),
            buf.data_ptr())
    if refused:
        with pytest.raises(hip().SealHipError, match="workspace too small"):
            ctx.rotate_accumulate(*args, wb - 1, stream())
    ctx.rotate_accumulate(*args, wb, stream())
    got = from_dev(out)
    for c in range(count):
        want = None
        for h, (e, k) in enumerate(zip(elts, keys)):
            rot = cts[h, c] if k is None else ck.apply_galois_keyswitch(scheme, cts[h, c], e, k, moduli, L, logn)
            want = rot if want is None else ck.mod_add(want, rot, moduli)
        np.testing.assert_array_equal(got[c], want, err_msg=f"ciphertext {c}")
    np.testing.assert_array_equal(from_dev(din), cts)


def test_rotate_sum_in_a_captured_graph():
    """The hoisted rotation sum waits for nothing on the host, so it can be captured: a
    captured call (with zero digits in the batch, so the fix runs) replays to the eager
    words three times, with eager work between the replays."""
    logn, n = 12, 1 << 12
    moduli = ck.coeff_modulus_create(n, [60, 40, 40, 60])
    L, count = 3, 2
    ctx = hip().Context(CKKS, n, moduli)
    rng = np.random.default_rng(41)
    cts = ck.uniform_residues(rng, (count, 2, L, n), moduli[:L])
    c1 = ck.ntt_rns(cts[1, 1], moduli[:L], logn, inverse=True)
    c1[:, 7] = 0
    cts[1, 1] = ck.ntt_rns(c1, moduli[:L], logn)
    steps = [1, 2, 5]
    elts = [ck.galois_elt(logn, s) for s in steps]
    keys = [ck.random_key(rng, moduli, logn) for _ in steps]
    dkeys = [to_dev(k) for k in keys]
    hb, hw = ctx.hoisted_key_size(L), ctx.hoisted_key_workspace_size(L)
    hws = ws(hw)
    hkeys = []
    for e, dk in zip(elts, dkeys):
        h = empty_dev(((hb + 7) // 8,))
        ctx.hoisted_key_prepare(dk.data_ptr(), e, L, h.data_ptr(), hws.data_ptr(), hw, stream())
        hkeys.append(h)
    din = to_dev(cts)
    out = empty_dev((count, 2, L, n))
    rw = ctx.rotate_sum_workspace_size(count, L)
    rws = ws(rw)
    hp, kp = [h.data_ptr() for h in hkeys], [k.data_ptr() for k in dkeys]
    ctx.rotate_sum(din.data_ptr(), count, L, elts, hp, kp, out.data_ptr(), rws.data_ptr(), rw, stream())
    eager = from_dev(out).copy()
    for c in range(count):
        want = None
        for e, k in zip(elts, keys):
            rot = ck.apply_galois_keyswitch(CKKS, cts[c], e, k, moduli, L, logn)
            want = rot if want is None else ck.mod_add(want, rot, moduli)
        np.testing.assert_array_equal(eager[c], want, err_msg=f"eager, ciphertext {c}")
    graph = torch.cuda.CUDAGraph()
    cap = torch.cuda.Stream()
    cap.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(graph, stream=cap):
        ctx.rotate_sum(din.data_ptr(), count, L, elts, hp, kp, out.data_ptr(), rws.data_ptr(), rw,
                       torch.cuda.current_stream().cuda_stream)
    torch.cuda.current_stream().wait_stream(cap)
    torch.cuda.synchronize()
    other = empty_dev((count, 2, L, n))
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(from_dev(out), eager, err_msg="replay")
        # eager work between replays, on the same workspace
        ctx.rotate_sum(din.data_ptr(), count, L, elts, hp, kp, other.data_ptr(), rws.data_ptr(), rw, stream())
        torch.cuda.synchronize()
        np.testing.assert_array_equal(from_dev(other), eager, err_msg="eager between replays")


def test_hoisted_key_bound_to_level_and_element():
    """A prepared key names its level and Galois element; using it at another level or
    for another element is an invalid argument, not wrong words."""
    logn, n = 12, 1 << 12
    moduli = ck.coeff_modulus_create(n, [60, 40, 40, 60])
    K = len(moduli)
    ctx = hip().Context(CKKS, n, moduli)
    rng = np.random.default_rng(3)
    key = to_dev(ck.random_key(rng, moduli, logn))
    e1, e2 = ck.galois_elt(logn, 1), ck.galois_elt(logn, 2)
    L = 3
    hb, hw = ctx.hoisted_key_size(L), ctx.hoisted_key_workspace_size(L)
    h = empty_dev(((hb + 7) // 8,))
    ctx.hoisted_key_prepare(key.data_ptr(), e1, L, h.data_ptr(), ws(hw).data_ptr(), hw, stream())
    for lvl, elt in ((L, e2), (L - 1, e1)):
        din = to_dev(ck.uniform_residues(rng, (1, 2, lvl, n), moduli[:lvl]))
        out = empty_dev((1, 2, lvl, n))
        rw = ctx.rotate_sum_workspace_size(1, lvl)
        with pytest.raises(hip().SealHipError, match="prepared for another level"):
            ctx.rotate_sum(din.data_ptr(), 1, lvl, [elt], [h.data_ptr()], [key.data_ptr()], out.data_ptr(),
                           ws(rw).data_ptr(), rw, stream())
    # the matching level and element still work
    din = to_dev(ck.uniform_residues(rng, (1, 2, L, n), moduli[:L]))
    out = empty_dev((1, 2, L, n))
    rw = ctx.rotate_sum_workspace_size(1, L)
    ctx.rotate_sum(din.data_ptr(), 1, L, [e1], [h.data_ptr()], [key.data_ptr()], out.data_ptr(), ws(rw).data_ptr(),
                   rw, stream())
    want = ck.apply_galois_keyswitch(CKKS, from_dev(din)[0], e1, from_dev(key), moduli, L, logn)
    np.testing.assert_array_equal(from_dev(out)[0], want)


def test_rotate_sum_seven_rotations_two_passes():
    """Seven rotations: two passes of the hoisted products (4 + 3) accumulate into the
    output and reuse the product buffers."""
    run_case(CKKS, 12, [60, 40, 40, 60], 3, 3, [1, 2, 3, 5, -1, -4, 7], seed=77)
