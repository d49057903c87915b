"""Single key switches whose ModUp ends inside the key product: the residues of ModUp, hoisted sum and ModDown called one after the other, which
other tests compare with the oracle."""
import pytest

from __graft_entry__ import load_package
from test_gpu_rows_in_sum import residues

pytestmark = pytest.mark.gpu


# one, two and three digits, the last one short or the only one; all limbs of a digit below the level; both arithmetics; sums on both sides of
# the lines of the ModDown's split; 64 converted limbs of 2^13 (one launch: the general path), four digits and rings of one launch (ditto)
@pytest.mark.parametrize("log_n,chain,special,dnum,bits,nq", [
    (13, 6, 2, 3, 42, 6), (13, 6, 2, 3, 42, 2), (13, 6, 2, 3, 42, 5), (13, 4, 4, 1, 60, 3), (13, 24, 8, 3, 60, 24), (14, 7, 3, 3, 60, 7), (14, 5, 3, 2, 42, 4),
    (15, 8, 2, 4, 42, 8), (15, 9, 5, 2, 60, 9), (16, 13, 4, 3, 42, 13), (16, 13, 4, 3, 42, 1), (16, 2, 1, 2, 60, 2), (16, 24, 8, 3, 60, 17), (12, 6, 2, 3, 42, 6)])
def test_single_switches(log_n, chain, special, dnum, bits, nq):
    import torch
    pkg = load_package()
    N = 1 << log_n
    big = pkg.primes_below(60, log_n, chain + special)
    qs, ps = (big[:chain] if bits == 60 else big[:1] + pkg.primes_below(bits, log_n, chain - 1)), big[chain:]
    ctx = pkg.Context(log_n, qs, ps, dnum)
    gen = torch.Generator(device="cuda").manual_seed(nq)
    ct, key = residues(qs[:nq], (3,), N, gen), residues(qs + ps, (dnum, 2), N, gen)
    q = torch.tensor(qs[:nq], dtype=torch.int64, device="cuda").view(-1, 1)
    g = pow(5, 77, 2 * N)

    def composed(a, b):
        ext = ctx.modup_batch(a.contiguous()[None], nq)[0]
        return ctx.moddown_batch(ctx.hoisted_terms([[(ext, b.contiguous(), key, None, 1)]], nq), nq, 0)[0]

    zero = torch.zeros_like(ct[0])
    plain = composed(ct[2], zero)
    assert torch.equal(ctx.keyswitch(ct[2].contiguous(), key, nq), plain)
    assert torch.equal(ctx.keyswitch(ct[2].contiguous(), key, nq, ct[0].contiguous()), composed(ct[2], ct[0]))
    assert torch.equal(ctx.relinearize(ct, key, nq), (plain + ct[:2]) % q)
    for galois in (g, 2 * N - 1):
        turned = ctx.automorphism(ct[:2].contiguous(), galois, nq)
        want = composed(turned[1], turned[0])
        assert torch.equal(ctx.rotate(ct[:2].contiguous(), key, galois, nq), want)
        # a result in its operand's place; an operand at an odd word
        own = ct[:2].clone()
        assert torch.equal(ctx.rotate(own, key, galois, nq, out=own), want)
        odd = torch.empty(2 * nq * N + 1, dtype=torch.int64, device="cuda")[1:].view(2, nq, N)
        odd.copy_(ct[:2])
        if galois == g:
            assert torch.equal(ctx.rotate(odd, key, galois, nq), want)
