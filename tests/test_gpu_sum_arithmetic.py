"""Hoisted sums over primes of every size, one to four digits and every kind of term, against the oracle: integers take products in
pieces for up to three digits and primes below 2^60, and a general path beyond either."""
import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle import oracle as O

pytestmark = pytest.mark.gpu
LOG_N, SHIFT = 10, 3
N = 1 << LOG_N


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int64)).cuda()


@pytest.mark.parametrize("bits", [45, 52, 59, 60, 61])
@pytest.mark.parametrize("chain,dnum", [(3, 1), (4, 2), (6, 3), (4, 4)])
@pytest.mark.parametrize("largest", [False, True])
def test_every_kind_of_term(bits, chain, dnum, largest):
    """largest: every operand q - 1, the largest values that any step of the sums sees"""
    pkg = load_package()
    primes = pkg.primes_below(bits, LOG_N, chain + 2)
    qs, ps = primes[:chain], primes[chain:]
    orc, ctx, nq = O.Oracle(LOG_N, qs, ps, dnum), pkg.Context(LOG_N, qs, ps, dnum), chain
    rng = np.random.default_rng(bits * 10 + dnum)

    def residues(mods, lead, runs=1):
        out = np.empty(tuple(lead) + (len(mods), N), dtype=np.uint64)
        for j, q in enumerate(mods):
            out[..., j, :] = q - 1 if largest else np.repeat(rng.integers(0, q, tuple(lead) + (N // runs,), dtype=np.uint64), runs, axis=-1)
        return out

    ext = [residues(primes, (ctx.beta(nq),)) for _ in range(2)]
    b = [residues(qs, ()) for _ in range(2)]
    a = residues(qs, ())
    keys = [residues(primes, (dnum, 2)) for _ in range(2)]
    full, runs = [residues(primes, ()) for _ in range(2)], [residues(primes, (), 1 << SHIFT) for _ in range(2)]
    pt = O.Pt(residues(primes, ()), 1.0)
    d_ext, d_b, d_a, d_keys, d_full, d_pt = [dev(e) for e in ext], [dev(x) for x in b], dev(a), [dev(k) for k in keys], [dev(m) for m in full], dev(pt.data)
    d_runs = [ctx.compact_mask(dev(m), SHIFT) for m in runs]
    g1, g2 = pow(5, 7, 2 * N), pow(5, 100, 2 * N)
    # (source, b, key, mask kind and number, automorphism, with the plaintext factor)
    two = lambda kind, k, g, p: [(0, 0, k, (kind, 0), g, p), (1, 1, k, (kind, 1), g, p)]
    one = lambda mask, k, g, p, bb=0: [(0, bb, k, mask, g, p)]
    none = lambda mask, p: [(None, 1, None, mask, 1, p)]
    groups = [two("full", 0, g1, False), two("runs", 0, g1, False), two("runs", 1, g2, True), two("full", 1, g2, True),
              one(None, 0, g1, False), one(None, 0, g2, False, None), one(("full", 0), 1, g1, False), one(("runs", 1), 1, g2, False),
              one(None, 0, g1, True), one(("full", 1), 0, g1, True), none(None, False), none(("full", 0), False), none(None, True),
              # long enough for every running sum to be reduced on the way
              sum((two("runs", t % 2, g1 if t % 3 else g2, t % 2 == 1) + one(None, t % 2, g2, False) + none(None, False) for t in range(7)), [])]
    give, want = [], np.zeros((len(groups), 2, nq + 2, N), dtype=np.uint64)
    for o, terms in enumerate(groups):
        give.append([])
        for src, bb, k, mask, g, p in terms:
            m = None if mask is None else O.Pt((full if mask[0] == "full" else runs)[mask[1]], 1.0)
            d_m = None if mask is None else (d_full if mask[0] == "full" else d_runs)[mask[1]]
            shift = SHIFT if mask is not None and mask[0] == "runs" else 0
            factor = orc.ext_plain_product(m, pt, g2) if p else m
            give[-1].append((d_a if k is None else d_ext[src], d_b[bb] if bb is not None else None, d_keys[k] if k is not None else None, d_m,
                             g, shift, d_pt if p else None, g2))
            if k is None:
                y = orc.hoisted_sum([(a, b[bb], ("none",), factor)], nq)
            else:
                y = np.zeros((2, nq + 2, N), dtype=np.uint64)
                orc.L.orc_hoisted_term(orc.h, O._p(ext[src]), O._p(b[bb]) if bb is not None else None, O._p(keys[k]),
                                       O._p(np.ascontiguousarray(factor.data)) if factor is not None else None, g, nq, O._p(y), 0)
            want[o] = add(want[o], y, primes)
    give = [[t if t[6] is not None else t[:6] for t in terms] for terms in give]
    got = ctx.hoisted_terms(give, nq).cpu().numpy().view(np.uint64)
    for o in range(len(groups)):
        assert np.array_equal(got[o], want[o]), o
    # the longest sum by itself and many times over: few enough workgroups for its terms to be dealt to four, resp. two, groups of wavefronts
    for copies in (1, 520 // (2 * len(primes))):
        got = ctx.hoisted_terms(give[-1:] * copies, nq).cpu().numpy().view(np.uint64)
        assert all(np.array_equal(y, want[-1]) for y in got), copies


def add(x, y, primes):
    q = np.array(primes, dtype=np.uint64).reshape(-1, 1)
    s = x + y               # below 2^62
    return np.where(s >= q, s - q, s)
