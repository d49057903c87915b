"""GPU parity of the register-blocked transforms on every ring size they serve: whole key switches and rescales through
their fused forms, and batches on both sides of the line between the one-launch and the two-launch kernels."""
import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle import oracle as O
from oracle.oracle import _p

pytestmark = pytest.mark.gpu


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int64)).cuda()


def host(t):
    return t.cpu().numpy().view(np.uint64)


def top_and_random(rng, mods, lead, N):
    """random residues, the largest one in the first polynomial's first half"""
    out = np.empty(tuple(lead) + (len(mods), N), dtype=np.uint64)
    for j, q in enumerate(mods):
        out[..., j, :] = rng.integers(0, q, tuple(lead) + (N,), dtype=np.uint64)
        out.reshape(-1, len(mods), N)[0, j, : N // 2] = q - 1
    return out


# digits of 1, 2, 5, 8 limbs take a kernel each; of 9 the forms without a fused conversion
@pytest.mark.parametrize("log_n", [10, 11, 12, 13, 14, 15])
@pytest.mark.parametrize("chain,special,dnum", [(3, 1, 3), (6, 2, 3), (10, 4, 2), (8, 5, 1), (9, 6, 1)])
def test_keyswitch_forms(log_n, chain, special, dnum):
    pkg = load_package()
    qs, ps = O.ckks_chain(log_n, chain, special)
    ctx, orc, N = pkg.Context(log_n, qs, ps, dnum), O.Oracle(log_n, qs, ps, dnum), 1 << log_n
    rng = np.random.default_rng(log_n * 100 + chain)
    key = top_and_random(rng, qs + ps, (dnum, 2), N)
    for nq in (chain, max(2, chain - 1)):
        ct = top_and_random(rng, qs[:nq], (3,), N)
        g = pow(5, 3, 2 * N)
        rot = np.empty((2, nq, N), dtype=np.uint64)
        for p in range(2):
            for j in range(nq):
                orc.L.orc_automorphism_ntt(orc.h, _p(ct[p, j]), _p(rot[p, j]), g)
        kb, ka = orc.keyswitch(rot[1], key)
        want = np.stack([orc.add_residues(rot[0], kb), ka])
        assert np.array_equal(host(ctx.rotate(dev(ct[:2]), dev(key), g, nq)), want)
        kb, ka = orc.keyswitch(ct[2], key)
        want = np.stack([orc.add_residues(ct[0], kb), orc.add_residues(ct[1], ka)])
        assert np.array_equal(host(ctx.relinearize(dev(ct), dev(key), nq)), want)
        want = np.empty((3, nq - 1, N), dtype=np.uint64)
        for p in range(3):
            orc.L.orc_rescale(orc.h, _p(ct[p]), nq, _p(want[p]))
        assert np.array_equal(host(ctx.rescale(dev(ct), nq)), want)


# limbs on both sides of where a ring goes over to one launch, and a run of polynomials that is cut
@pytest.mark.parametrize("log_n,polys,limbs", [(11, 1, 1), (12, 3, 5), (13, 21, 3), (13, 32, 2), (14, 19, 5), (14, 16, 6), (15, 7, 3),
                                               (15, 300, 3)])
def test_batches(log_n, polys, limbs):
    pkg = load_package()
    mods = [O.primes_below(61, log_n, 1)[0], O.primes_below(60, log_n, 1)[0]] + O.primes_below(44, log_n, 4)
    mods = mods[:limbs]
    ctx, orc, N = pkg.Context(log_n, mods, [], 1), O.Oracle(log_n, mods, [], 1, threads=8), 1 << log_n
    rng = np.random.default_rng(log_n + polys)
    a = top_and_random(rng, mods, (polys,), N)
    idx = list(range(len(mods)))
    for inverse in (False, True):
        d = dev(a)
        ctx.ntt(d, idx, inverse=inverse)
        got = host(d)
        for p in sorted({0, polys // 2, polys - 1}):
            want = a[p].copy()
            orc.ntt(want, idx, inverse=inverse)
            assert np.array_equal(got[p], want), (inverse, p)
        ctx.ntt(d, idx, inverse=not inverse)
        assert np.array_equal(host(d), a)


@pytest.mark.parametrize("log_n,polys", [(12, 2), (13, 5), (13, 24), (14, 24), (15, 3)])
@pytest.mark.parametrize("drop", [0, 1])
def test_moddown_of_batches(log_n, polys, drop):
    pkg = load_package()
    qs, ps = O.ckks_chain(log_n, 6, 3)
    ctx, orc, N, nq = pkg.Context(log_n, qs, ps, 2), O.Oracle(log_n, qs, ps, 2), 1 << log_n, 5
    rng = np.random.default_rng(log_n + polys + drop)
    y = top_and_random(rng, qs[:nq] + ps, (polys,), N)
    got = host(ctx.moddown_batch(dev(y), nq, drop))
    for p in sorted({0, polys // 2, polys - 1}):
        want = np.empty((nq - drop, N), dtype=np.uint64)
        orc.L.orc_moddown_drop(orc.h, _p(y[p].copy()), nq, drop, _p(want))
        assert np.array_equal(got[p], want), p


# limbs on both sides of where a pass gives a thread eight points instead of sixteen (2^16 points: 32 limbs for columns, 40 for
# rows; 2^13: 256 and 320, out of a launch that would be one), primes of all three arithmetic forms, extreme residues
@pytest.mark.parametrize("log_n,polys,limbs", [(16, 1, 1), (16, 2, 16), (16, 3, 11), (16, 4, 10), (16, 1, 41), (15, 3, 27), (14, 5, 19)])
@pytest.mark.parametrize("bits", [42, 60, 61])
def test_points_per_thread(log_n, polys, limbs, bits):
    import torch
    pkg = load_package()
    primes = O.primes_below(bits, log_n, limbs)
    ctx, orc, N = pkg.Context(log_n, primes, [], 1), O.Oracle(log_n, primes, [], 1), 1 << log_n
    rng = np.random.default_rng(log_n * 1000 + polys * limbs + bits)
    a = top_and_random(rng, primes, (polys,), N)
    d = dev(a)
    ctx.ntt(d, list(range(limbs)))
    got = host(d)
    for p in {0, polys - 1}:   # the oracle takes its time: the first and the last polynomial, the others by the way back
        want = a[p].copy()
        orc.ntt(want, list(range(limbs)))
        assert np.array_equal(got[p], want)
    ctx.ntt(d, list(range(limbs)), inverse=True)
    assert torch.equal(d, dev(a))


# term counts around the four products between reductions and the 64 terms of the double-precision sums, in the lists that
# travel in the kernel arguments (up to 32 terms) and in those that do not; unmasked terms, masks through an automorphism
@pytest.mark.parametrize("n_terms", [1, 3, 4, 5, 32, 33, 64, 65, 129])
def test_masked_sum_lengths(n_terms):
    pkg = load_package()
    log_n, g = 10, 25
    mods = [O.primes_below(60, log_n, 1)[0], O.primes_below(44, log_n, 1)[0]]
    ctx, orc, N = pkg.Context(log_n, mods, [], 1), O.Oracle(log_n, mods, [], 1), 1 << log_n
    rng = np.random.default_rng(n_terms)
    cts, masks = top_and_random(rng, mods, (3, 2), N), top_and_random(rng, mods, (2,), N)
    masks[0, :, : N // 2] = np.array(mods, dtype=np.uint64)[:, None] - np.uint64(1)
    turned = np.empty_like(masks)
    for i in range(2):
        for j in range(2):
            orc.L.orc_automorphism_ntt(orc.h, _p(masks[i, j]), _p(turned[i, j]), g)
    dct, dmask = [dev(c) for c in cts], [dev(m) for m in masks]
    spec = [(t % 3, None if t % 7 == 3 else t % 2, g if t % 5 == 4 else 0) for t in range(n_terms)]
    got = host(ctx.masked_sum_batch([[(dct[c], None if m is None else dmask[m], gal if m is not None else 0) for c, m, gal in spec]], 2, 2))
    want = np.zeros((2, 2, N), dtype=object)
    for c, m, gal in spec:
        want += cts[c].astype(object) * (1 if m is None else (turned if gal else masks)[m].astype(object))
    want %= np.array(mods, dtype=object)[:, None]
    assert np.array_equal(got[0], want.astype(np.uint64))


def random_residues(ctx, gen, lead, N):
    import torch
    q = torch.tensor(ctx.q, dtype=torch.int64, device="cuda").view(-1, 1)
    return torch.randint(0, 1 << 62, tuple(lead) + (len(ctx.q), N), dtype=torch.int64, device="cuda", generator=gen).remainder_(q)


# lists without a term that has no mask, lists of such terms alone, and both mixed, take two kernels
@pytest.mark.parametrize("n_polys", [1, 2, 3])
@pytest.mark.parametrize("n_terms", [1, 5, 33, 65])
@pytest.mark.parametrize("masked", ["all", "none", "every second"])
def test_masked_sum_with_and_without_masks(n_polys, n_terms, masked):
    pkg = load_package()
    log_n, N, g = 11, 1 << 11, pow(5, 7, 1 << 12)
    mods = [O.primes_below(60, log_n, 1)[0], O.primes_below(44, log_n, 1)[0]]
    ctx, orc = pkg.Context(log_n, mods, [], 1), O.Oracle(log_n, mods, [], 1)
    rng = np.random.default_rng(100 * n_terms + n_polys)
    cts, masks = top_and_random(rng, mods, (3, n_polys), N), top_and_random(rng, mods, (2,), N)
    turned = np.empty_like(masks)
    for i in range(2):
        for j in range(2):
            orc.L.orc_automorphism_ntt(orc.h, _p(masks[i, j]), _p(turned[i, j]), g)
    dct, dmask = [dev(c) for c in cts], [dev(m) for m in masks]
    outs, want = [], []
    for o in range(2):
        spec = [((t + o) % 3, t % 2 if masked == "all" or (masked != "none" and t % 2 == o) else None, g if t % 3 == 2 else 0) for t in range(n_terms)]
        outs.append([(dct[c], None if m is None else dmask[m], gal) for c, m, gal in spec])   # an automorphism without a mask: no effect
        w = np.zeros((n_polys, 2, N), dtype=object)
        for c, m, gal in spec:
            w += cts[c].astype(object) * (1 if m is None else (turned if gal else masks)[m].astype(object))
        want.append((w % np.array(mods, dtype=object)[:, None]).astype(np.uint64))
    got = host(ctx.masked_sum_batch(outs, 2, n_polys))
    assert np.array_equal(got, np.stack(want))


# A term without a mask is an addition of what it reads: two polynomials where a masked term reads three, 0.69 of the time
# measured on this list.  The line is halfway to the 0.98 of a sum that multiplies by one and reads a third.
def test_masked_sum_without_masks_reads_none():
    import torch
    pkg = load_package()
    log_n, n_terms = 13, 128
    ctx = pkg.Context(log_n, O.primes_below(60, log_n, 6), [], 1)
    gen = torch.Generator(device="cuda").manual_seed(1)
    cts = [random_residues(ctx, gen, (2,), 1 << log_n) for _ in range(n_terms)]
    masks = [random_residues(ctx, gen, (), 1 << log_n) for _ in range(n_terms)]
    lists = {"masked": [list(zip(cts, masks))], "plain": [[(c, None) for c in cts]]}
    best = dict.fromkeys(lists, float("inf"))
    for _ in range(8):   # both in turn
        for name, groups in lists.items():
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(10):
                ctx.masked_sum_batch(groups, 6, 2)
            end.record()
            torch.cuda.synchronize()
            best[name] = min(best[name], start.elapsed_time(end))
    assert best["plain"] < 0.84 * best["masked"], best
