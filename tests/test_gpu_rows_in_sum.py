"""Hoisted sums whose dropped limbs leave as the first pass of the ModDown's inverse transform (hemm_hoisted_moddown, key switches):
the residues of the sum and the ModDown called one after the other, which other tests compare with the oracle."""
import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def residues(primes, lead, N, gen):
    import torch
    q = torch.tensor(primes, dtype=torch.int64, device="cuda").view(-1, 1)
    return torch.randint(0, 1 << 62, tuple(lead) + (len(primes), N), dtype=torch.int64, device="cuda", generator=gen).remainder_(q)


# rings of two launches, a ring that goes over to one (2^13 with 64 dropped limbs or more), one that never has two (2^12); sums of one
# launch and, from 16384 workgroups on, of one per kind of limb; more than six digits (limbs below 2^44 summed as integers); term
# lists in the arguments and, with more than 32 terms, in memory; 42-bit and 60-bit limbs dropped beside the special ones
@pytest.mark.parametrize("log_n,chain,special,dnum,bits,n_out,terms", [
    (12, 4, 2, 2, 42, 2, 1), (13, 3, 1, 3, 42, 1, 1), (13, 5, 2, 5, 42, 2, 3), (13, 5, 2, 1, 42, 16, 1), (13, 8, 2, 8, 42, 2, 2),
    (14, 6, 3, 2, 60, 3, 1), (14, 4, 2, 2, 61, 2, 1), (15, 4, 2, 2, 42, 5, 7), (16, 2, 1, 1, 42, 1, 1), (16, 7, 4, 3, 42, 2, 17), (16, 7, 4, 3, 42, 12, 1)])
@pytest.mark.parametrize("drop", [0, 1])
@pytest.mark.parametrize("compact", [False, True])
def test_rows_in_sum(log_n, chain, special, dnum, bits, n_out, terms, drop, compact):
    import torch
    pkg = load_package()
    if compact and dnum > 6:
        pytest.skip("compact keys take at most six digits")
    N, nq = 1 << log_n, chain
    big = pkg.primes_below(61 if bits == 61 else 60, log_n, chain + special)
    qs = big[:chain] if bits >= 60 else big[:1] + pkg.primes_below(bits, log_n, chain - 1)
    ps = big[chain:]
    ctx = pkg.Context(log_n, qs, ps, dnum)
    gen = torch.Generator(device="cuda").manual_seed(log_n * 100 + n_out)
    beta = ctx.beta(nq)
    ext, b = residues(qs + ps, (2, beta), N, gen), residues(qs, (2,), N, gen)
    keys = [residues(qs + ps, (dnum, 2), N, gen) for _ in range(2)]
    mask = residues(qs + ps, (), N, gen)
    give = [ctx.compact_key(k) for k in keys] if compact else keys
    groups = [[(ext[(o + t) % 2], b[t % 2], give[t % 2], mask if t % 3 == 1 else None, pow(5, 3 * o + t, 2 * N)) for t in range(terms)]
              for o in range(n_out)]
    want = ctx.moddown_batch(ctx.hoisted_terms(groups, nq, compact_keys=compact), nq, drop)
    assert torch.equal(ctx.hoisted_moddown(groups, nq, drop, compact_keys=compact), want)


@pytest.mark.parametrize("log_n", [13, 16])
@pytest.mark.parametrize("pattern", ["all", "even", "first half of a row"])
def test_rows_in_sum_of_the_largest_residues(log_n, pattern):
    """A sum that is q - 1 at every, or at every second, place: the largest values the row pass adds up and multiplies, in double
    precision for the largest prime below 2^44 that there is."""
    import torch
    pkg = load_package()
    N = 1 << log_n
    big = pkg.primes_below(60, log_n, 2)
    qs, ps = big[:1] + pkg.primes_below(44, log_n, 2), big[1:]
    ctx = pkg.Context(log_n, qs, ps, 1)
    q = torch.tensor(qs + ps, dtype=torch.int64, device="cuda").view(-1, 1)
    n = torch.arange(N, device="cuda")
    at = {"all": n >= 0, "even": n % 2 == 0, "first half of a row": n % 256 < 128}[pattern]
    ext = torch.where(at, q - 1, torch.zeros_like(q)).unsqueeze(0).contiguous()
    key = torch.ones((1, 2, 4, N), dtype=torch.int64, device="cuda")
    groups = [[(ext, None, key, None, 1)]]
    for drop in (0, 1):
        y = ctx.hoisted_terms(groups, 3)
        assert bool((y[0, 1] == ext[0]).all())
        assert torch.equal(ctx.hoisted_moddown(groups, 3, drop), ctx.moddown_batch(y, 3, drop))
