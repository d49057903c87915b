"""ModDowns of 2^16 points whose inverse column pass, conversion and forward column pass are one kernel (two to five sources, by the number of
polynomials and targets) against the four launches, which calls of four polynomials take, and the oracle.  Every polynomial holds data of its own."""
import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle import oracle as O
from test_gpu_rows_in_sum import moddown_to, residues

pytestmark = pytest.mark.gpu
LOG_N, N = 16, 1 << 16


def chain(bits, sources, targets):
    """Primes of a ModDown with rescale: the last chain prime and the special ones are dropped."""
    pkg = load_package()
    p = pkg.primes_below(50 if bits == 50 else 60, LOG_N, sources + targets)
    ps = p[:sources - 1]
    return (pkg.primes_below(42, LOG_N, targets + 1) if bits == 42 else p[sources - 1:]), ps


def four_launches(ctx, y, nq, drop):
    import torch
    return torch.cat([ctx.moddown_batch(part.clone(), nq, drop) for part in y.split(4)])


# numbers of polynomials on both sides of each line: eight; nine to eleven; one round of sixteen and the next; last rounds of few; a batch cut into runs
# (5 -> 8 from 57 polynomials: 48 + 9, 48 + 16, 56 + 44; 5 -> 12 from 38: 32 + 16, 32 + 31)
@pytest.mark.parametrize("bits,sources,targets,polys", [
    (42, 2, 5, (7, 8, 9, 10, 33)), (60, 2, 12, (12, 13, 16, 17)), (42, 3, 6, (8, 9, 11, 12, 17)), (50, 3, 7, (12, 13, 16, 17)), (60, 4, 7, (8, 12, 19, 20)),
    (50, 4, 7, (12, 13, 23, 24)), (42, 5, 8, (7, 8, 12, 13, 56, 57, 64, 100)), (50, 5, 8, (20, 24, 26)), (60, 5, 9, (16, 17, 29, 30, 40)),
    (42, 5, 12, (28, 32, 40, 48, 63)), (42, 5, 13, (16,)), (42, 6, 5, (16,))])
def test_batches(bits, sources, targets, polys):
    import torch
    qs, ps = chain(bits, sources, targets)
    ctx, orc, nq = load_package().Context(LOG_N, qs, ps, 3), O.Oracle(LOG_N, qs, ps, 3), targets + 1
    y = residues(qs + ps, (max(polys),), N, torch.Generator(device="cuda").manual_seed(sources * 100 + targets))
    y[0], y[1] = torch.tensor(qs + ps, device="cuda").view(-1, 1) - 1, 0
    want = four_launches(ctx, y, nq, True)
    few = [0, max(polys) - 1]
    assert np.array_equal(want[few].cpu().numpy().view(np.uint64), orc.moddown_drop(y[few].cpu().numpy().view(np.uint64), nq, True))
    for n in polys:
        got = ctx.moddown_batch(y[:n].clone(), nq, True)
        assert torch.equal(got, want[:n]), n
        del got
        if sources in (4, 5):
            assert torch.equal(ctx.moddown_batch(y[:n].clone(), nq, True, column_slab=True), want[:n]), n


# results in a list: rows of the dropped limbs made by the sum, one run and (5 -> 8, 64 polynomials; results on odd places take the sum whole) two
@pytest.mark.parametrize("bits", [42, 60])
@pytest.mark.parametrize("n_out,targets", [(4, 7), (16, 8), (32, 8), (20, 12), (24, 12)])
def test_under_sums(bits, n_out, targets):
    import torch
    pkg = load_package()
    qs, ps = chain(bits, 5, targets)
    ctx, nq = pkg.Context(LOG_N, qs, ps, 3), targets + 1
    gen = torch.Generator(device="cuda").manual_seed(n_out)
    ext, b, key = residues(qs + ps, (ctx.beta(nq),), N, gen), residues(qs, (), N, gen), residues(qs + ps, (3, 2), N, gen)
    groups = [[(ext, b, key, None, pow(5, 3 * o + 1, 2 * N))] for o in range(n_out)]
    sums = ctx.hoisted_terms(groups, nq)
    want = four_launches(ctx, sums.view(2 * n_out, nq + 4, N), nq, True).view(n_out, 2, targets, N)
    assert torch.equal(ctx.hoisted_moddown(groups, nq, True), want)
    for pad in (2, 1):
        got, guard = moddown_to(pkg, ctx, groups, nq, 1, False, targets * N + pad)
        assert torch.equal(got, want) and bool((guard == -1).all())
