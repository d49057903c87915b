"""Hoisted sums that share launches with the ModDown behind them (hemm_hoisted_moddown, hemm_hoisted_moddown_to, key switches): dropped
limbs leave as the first pass of their inverse transform, kept ones are summed under the last pass of the forward transform.  The
residues are those of the sum and the ModDown called one after the other, which other tests compare with the oracle."""
import ctypes

import pytest

from __graft_entry__ import load_package

pytestmark = pytest.mark.gpu


def residues(primes, lead, N, gen):
    import torch
    q = torch.tensor(primes, dtype=torch.int64, device="cuda").view(-1, 1)
    return torch.randint(0, 1 << 62, tuple(lead) + (len(primes), N), dtype=torch.int64, device="cuda", generator=gen).remainder_(q)


# rings of two launches, a ring that goes over to one (2^13 with 64 dropped limbs or more), one that never has two (2^12); sums of one
# launch and, from 16384 workgroups on, of one per kind of limb; more than six digits (limbs below 2^44 summed as integers); term
# lists in the arguments and, with more than 32 terms, in memory; 42-bit and 60-bit limbs dropped beside the special ones.  Kept limbs are
# summed under the ModDown's last pass from 1024 workgroups with two terms an output at most, from 4096 with more: both sides of
# either line, a kernel for each kind of limb there too, more results than one list holds, a conversion too wide for it
@pytest.mark.parametrize("log_n,chain,special,dnum,bits,n_out,terms", [
    (12, 4, 2, 2, 42, 2, 1), (13, 3, 1, 3, 42, 1, 1), (13, 5, 2, 5, 42, 2, 3), (13, 5, 2, 1, 42, 16, 1), (13, 8, 2, 8, 42, 2, 2),
    (14, 6, 3, 2, 60, 3, 1), (14, 4, 2, 2, 61, 2, 1), (15, 4, 2, 2, 42, 5, 7), (16, 2, 1, 1, 42, 1, 1), (16, 7, 4, 3, 42, 2, 17), (16, 7, 4, 3, 42, 12, 1),
    (14, 6, 3, 2, 60, 8, 2), (15, 5, 2, 3, 42, 3, 1), (15, 5, 2, 3, 42, 4, 3), (15, 5, 2, 3, 42, 10, 3), (16, 7, 4, 3, 42, 32, 1),
    (16, 2, 1, 1, 42, 33, 1), (16, 8, 1, 8, 42, 2, 1), (15, 9, 9, 1, 60, 2, 1)])
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
    # (two results at a time: in more launches than a larger batch on 2^16 points takes)
    want = torch.cat([ctx.moddown_batch(y, nq, drop) for y in ctx.hoisted_terms(groups, nq, compact_keys=compact).split(2)])
    assert torch.equal(ctx.hoisted_moddown(groups, nq, drop, compact_keys=compact), want)
    # results apart from each other, 16 bytes and 8 bytes aligned
    for pad in (2, 1):
        got, guard = moddown_to(pkg, ctx, groups, nq, drop, compact, (nq - drop) * N + pad)
        assert torch.equal(got, want) and bool((guard == -1).all())


def moddown_to(pkg, ctx, groups, nq, drop, compact, stride, room=None):
    """hemm_hoisted_moddown_to with result o in row n_out - 1 - o of a buffer: (results, the words behind each polynomial)"""
    import torch
    flat, N, n_out, nq_out = [t for g in groups for t in g], ctx.N, len(groups), nq - drop
    arr = (pkg.RotTerm * len(flat))()
    for i, (e, bb, k, m, g) in enumerate(flat):
        arr[i] = pkg.RotTerm(e.data_ptr(), bb.data_ptr() if bb is not None else None, k.data_ptr(), m.data_ptr() if m is not None else None, g, 0,
                             None, 1, int(compact))
    offs = [0]
    for g in groups:
        offs.append(offs[-1] + len(g))
    if room is None:
        room = torch.full((n_out, 2, stride), -1, dtype=torch.int64, device="cuda")
    outs = (ctypes.c_void_p * n_out)(*[room[n_out - 1 - o].data_ptr() for o in range(n_out)])
    y = torch.empty((n_out, 2, nq + ctx.nP, N), dtype=torch.int64, device="cuda")
    ws = torch.empty((n_out, 2, nq_out, N), dtype=torch.int64, device="cuda")
    pkg.check(pkg.lib().hemm_hoisted_moddown_to(ctx.h, arr, (ctypes.c_uint32 * len(offs))(*offs), n_out, nq, 0, drop, y.data_ptr(), outs, stride,
                                                ws.data_ptr(), None))
    r = room.flip(0)
    return r[:, :, : nq_out * N].reshape(n_out, 2, nq_out, N), r[:, :, nq_out * N:]


def test_results_that_replace_what_the_sum_reads():
    """Results in the memory of a b-polynomial, of the extended digits and of a key: read by the sum to its end, written at the end."""
    import torch
    pkg = load_package()
    log_n, nq = 16, 4
    N = 1 << log_n
    big = pkg.primes_below(60, log_n, 3)
    qs, ps = big[:1] + pkg.primes_below(42, log_n, 3), big[1:]
    ctx = pkg.Context(log_n, qs, ps, 2)
    gen = torch.Generator(device="cuda").manual_seed(9)
    key, ct = residues(qs + ps, (2, 2), N, gen), residues(qs, (2,), N, gen)
    g = pow(5, 7, 2 * N)
    want = ctx.rotate(ct, key, g, nq)
    assert torch.equal(ctx.rotate(ct.clone(), key, g, nq), want)
    own = ct.clone()
    ctx.rotate(own, key, g, nq, out=own)
    assert torch.equal(own, want)
    for victim in ("b", "ext", "key"):
        room = torch.empty((4, 2, 6 * N * 2), dtype=torch.int64, device="cuda")   # four results, each room for a whole operand
        ext, b = residues(qs + ps, (2,), N, gen), residues(qs, (), N, gen)
        groups = [[(ext, b, key, None, pow(5, 3 + o, 2 * N))] for o in range(4)]
        want = ctx.hoisted_moddown(groups, nq, 0)
        moved = {"b": b, "ext": ext, "key": key}
        flat = room[1].view(-1)[: moved[victim].numel()]
        flat.copy_(moved[victim].reshape(-1))
        moved[victim] = flat.view(moved[victim].shape)
        groups = [[(moved["ext"], moved["b"], moved["key"], None, pow(5, 3 + o, 2 * N))] for o in range(4)]
        got, _ = moddown_to(pkg, ctx, groups, nq, 0, False, 6 * N * 2, room)
        assert torch.equal(got, want), victim


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
