"""The inner sums of a plaintext product (hemm_diagonal_sums) by themselves, against sums of the oracle's hoisted terms: primes at both ends of
the two arithmetics, one to three digits, the fewest and the most baby steps and giant ones, runs wider and narrower than a wavefront's
residues, and every operand, key and table entry at q - 1, the largest values that any step of the lazy dot products sees."""
import ctypes

import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle import oracle as O

pytestmark = pytest.mark.gpu
LOG_N = 10
N = 1 << LOG_N
OUT = 8    # inner sums of a chunk of the tables, [limb][run][chunk][g][OUT] of 16 bytes
MASK30 = (1 << 30) - 1


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int64)).cuda()


@pytest.mark.parametrize("bits", [33, 44, 45, 60])
@pytest.mark.parametrize("chain, dnum, k, w, g", [(2, 1, 4, 4, 4), (4, 2, 8, 16, 8), (5, 3, 32, 32, 32), (5, 3, 64, 128, 8), (4, 2, 128, 256, 32)])
@pytest.mark.parametrize("largest", [False, True])
def test_diagonal_sums(bits, chain, dnum, k, w, g, largest):
    pkg = load_package()
    primes = pkg.primes_below(bits, LOG_N, chain + 2)
    qs, ps, E = primes[:chain], primes[chain:], chain + 2
    orc, ctx = O.Oracle(LOG_N, qs, ps, dnum), pkg.Context(LOG_N, qs, ps, dnum)
    rng = np.random.default_rng(bits * 1000 + chain * 10 + g)
    giants, runs = 2 * k // g, 2 * w
    chunks = -(-giants // OUT)

    def residues(mods, lead, n=N):
        out = np.empty(tuple(lead) + (len(mods), n), dtype=np.uint64)
        for j, q in enumerate(mods):
            out[..., j, :] = q - 1 if largest else rng.integers(0, q, tuple(lead) + (n,), dtype=np.uint64)
        return out

    def times(x, factors):   # x [..][limbs][n] times one number per limb
        f = np.array(factors, dtype=object).reshape(-1, 1)
        return (x.astype(object) * f % np.array(primes[: len(factors)], dtype=object).reshape(-1, 1)).astype(np.uint64)

    ext, a = residues(primes, (ctx.beta(chain),)), residues(qs, (2,))
    b, key = residues(qs, ()), residues(primes, (dnum, 2))
    entries = residues(primes, (giants, g), runs)
    entries[:, 0, chain:] = 0   # the rotation by nothing enters on the chain limbs
    table = np.zeros((E, runs, chunks, g, OUT, 4), dtype=np.uint32)
    shifted = times(entries, [1 << 30] * E)
    for t in range(giants):
        for i, part in enumerate((entries & MASK30, entries >> 30, shifted & MASK30, shifted >> 30)):
            table[:, :, t // OUT, :, t % OUT, i] = part[t].transpose(1, 2, 0)

    galois = [pow(5, j, 2 * N) for j in range(g)]
    P = [int(np.prod([p % q for p in ps], dtype=object)) % q for q in qs]

    def sums(b):
        y = np.zeros((giants, 2, E, N), dtype=np.uint64)
        for t in range(giants):
            factors = np.ascontiguousarray(np.repeat(entries[t], N // runs, axis=-1))
            for pol in (0, 1):
                y[t, pol, :chain] = (a[pol].astype(object) * factors[0, :chain].astype(object) % np.array(qs, dtype=object).reshape(-1, 1)).astype(np.uint64)
            for j in range(1, g):
                orc.L.orc_hoisted_term(orc.h, O._p(ext), O._p(b), O._p(key), O._p(factors[j]), galois[j], chain, O._p(y[t]), 1)
        return y

    f = pkg.lib().hemm_diagonal_sums
    vp, u32 = ctypes.c_void_p, ctypes.c_uint32
    f.argtypes = [vp, vp, vp, ctypes.c_size_t, u32, u32, u32, u32, ctypes.c_int, vp, vp, vp]
    words = ctypes.c_size_t()
    pkg.check(pkg.lib().hemm_diagonal_table_words(ctx.h, u32(k), u32(w), u32(g), u32(chain), ctypes.byref(words)))
    assert words.value * 8 == table.nbytes
    d_ext, d_a, d_key, d_table = dev(ext), dev(a), dev(key), dev(table.view(np.uint64))
    d_compact = ctx.compact_key(d_key)
    # with and without the factor P on b: the largest value of either is q - 1
    pairs = [(0, b, sums(b))]
    pairs.append((1, b, sums(times(b, [pow(p, -1, q) for p, q in zip(P, qs)]))) if largest else (1, times(b, P), pairs[0][2]))
    for pre, given, want in pairs:
        d_b = dev(given)
        for flags, key_of in ((0, d_key), (1, d_compact)):
            terms = (pkg.RotTerm * (g - 1))(*[pkg.RotTerm(d_ext.data_ptr(), d_b.data_ptr(), key_of.data_ptr(), None, galois[j], 0, None, 1, flags)
                                              for j in range(1, g)])
            y = dev(np.full((giants, 2, E, N), -1, dtype=np.int64))
            pkg.check(f(ctx.h, terms, d_a.data_ptr(), chain * N, k, w, g, chain, pre, d_table.data_ptr(), y.data_ptr(), None))
            assert np.array_equal(y.cpu().numpy().view(np.uint64), want), (pre, flags)


def test_a_residue_pair_lies_in_one_run():
    """Rows of N / 2 slots would have runs of one residue, where the sums take residues in pairs"""
    pkg = load_package()
    primes = pkg.primes_below(45, LOG_N, 4)
    ctx = pkg.Context(LOG_N, primes[:2], primes[2:], 1)
    words, u32 = ctypes.c_size_t(), ctypes.c_uint32
    for w, some in ((N // 4, True), (N // 2, False)):
        pkg.check(pkg.lib().hemm_diagonal_table_words(ctx.h, u32(4), u32(w), u32(4), u32(2), ctypes.byref(words)))
        assert (words.value != 0) == some
