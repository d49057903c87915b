"""Key products of more digits than one reduction takes (four), against the oracle: hoisted sums with one source and with two masked ones, and the
classic key switch; primes of 60 and 61 bits and small ones, random operands and every one at q - 1."""
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


@pytest.mark.parametrize("bits", [44, 60, 61])
@pytest.mark.parametrize("digits", [4, 5, 8, 9, 13])
@pytest.mark.parametrize("largest", [False, True])
def test_many_digits(bits, digits, largest):
    pkg = load_package()
    primes = pkg.primes_below(bits, LOG_N, digits + 2)
    qs, ps, nq = primes[:digits], primes[digits:], digits
    orc, ctx = O.Oracle(LOG_N, qs, ps, digits), pkg.Context(LOG_N, qs, ps, digits)
    rng = np.random.default_rng(bits * 100 + digits)

    def residues(mods, lead, runs=1):
        out = np.empty(tuple(lead) + (len(mods), N), dtype=np.uint64)
        for j, q in enumerate(mods):
            out[..., j, :] = q - 1 if largest else np.repeat(rng.integers(0, q, tuple(lead) + (N // runs,), dtype=np.uint64), runs, axis=-1)
        return out

    ext, b, key = [residues(primes, (digits,)) for _ in range(2)], [residues(qs, ()) for _ in range(2)], residues(primes, (digits, 2))
    full, runs = [residues(primes, ()) for _ in range(2)], [residues(primes, (), 1 << SHIFT) for _ in range(2)]
    d_ext, d_b, d_key = [dev(x) for x in ext], [dev(x) for x in b], dev(key)
    d_full, d_runs = [dev(m) for m in full], [ctx.compact_mask(dev(m), SHIFT) for m in runs]
    g = pow(5, 77, 2 * N)
    groups = [[(d_ext[0], d_b[0], d_key, None, g)],
              [(d_ext[i], d_b[i], d_key, d_full[i], g) for i in range(2)],
              [(d_ext[i], d_b[i], d_key, d_runs[i], g, SHIFT) for i in range(2)]]
    want = np.zeros((3, 2, nq + 2, N), dtype=np.uint64)
    for o, masks in enumerate(([None], full, runs)):
        for i, m in enumerate(masks):
            orc.L.orc_hoisted_term(orc.h, O._p(ext[i]), O._p(b[i]), O._p(key), O._p(m) if m is not None else None, g, nq, O._p(want[o]), 1)
    got = ctx.hoisted_terms(groups, nq).cpu().numpy().view(np.uint64)
    assert [np.array_equal(got[o], want[o]) for o in range(3)] == [True] * 3
    got = ctx.inner_product(d_ext[0], d_key, nq).cpu().numpy().view(np.uint64)
    acc = np.empty((2, nq + 2, N), dtype=np.uint64)
    orc.L.orc_inner_product(orc.h, O._p(ext[0]), O._p(key), nq, O._p(acc))
    assert np.array_equal(got, acc)
    p = residues(qs, ())
    got = ctx.keyswitch(dev(p), d_key, nq).cpu().numpy().view(np.uint64)
    ob, oa = np.empty((nq, N), dtype=np.uint64), np.empty((nq, N), dtype=np.uint64)
    orc.L.orc_keyswitch(orc.h, O._p(p), O._p(key), nq, O._p(ob), O._p(oa))
    assert np.array_equal(got, np.stack([ob, oa]))
