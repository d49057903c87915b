"""Primes on both sides of 2^60 - 2^27, where transforms and key switches change their arithmetic, against the oracle: operands at q - 1
and random ones."""
import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle import oracle as O

pytestmark = pytest.mark.gpu
LINE = 2**60 - 2**27


def dev(a):
    import torch
    return torch.from_numpy(np.array(a, order="C").view(np.int64)).cuda()


def host(t):
    return t.cpu().numpy().view(np.uint64)


def around_the_line(log_n):
    """The first primes above and at or below the line, and the first below 2^60."""
    step = 2 << log_n
    first = LINE // step * step + 1
    above = next(p for p in range(first if first > LINE else first + step, 2**60, step) if O.is_prime(p))
    below = next(p for p in range(first if first <= LINE else first - step, 0, -step) if O.is_prime(p))
    assert 2**60 - above < 2**27 <= 2**60 - below
    return [above, below, O.primes_below(60, log_n, 1)[0]]


def residues(rng, primes, lead, n, largest):
    out = np.empty(tuple(lead) + (len(primes), n), dtype=np.uint64)
    for j, q in enumerate(primes):
        out[..., j, :] = q - 1 if largest else rng.integers(0, q, tuple(lead) + (n,), dtype=np.uint64)
    return out


@pytest.mark.parametrize("log_n", [9, 10, 11, 12, 13, 14, 15, 16])
@pytest.mark.parametrize("polys", [1, 40])
def test_transforms(log_n, polys):
    qs = around_the_line(log_n)
    ctx, orc = load_package().Context(log_n, qs, [], 1), O.Oracle(log_n, qs, [], 1)
    rng, n = np.random.default_rng(log_n), 1 << log_n
    a = np.concatenate([residues(rng, qs, (1,), n, True), residues(rng, qs, (1,), n, False)])
    a[0, :, 1::2] = 0
    for inverse in (False, True):
        want = a.copy()
        orc.ntt(want, [0, 1, 2], inverse=inverse)
        for i in (0, 1):
            got = host(ctx.ntt(dev(np.broadcast_to(a[i], (polys,) + a[i].shape)), [0, 1, 2], inverse=inverse))
            assert np.array_equal(got, np.broadcast_to(want[i], got.shape)), (inverse, i)


# (2^15 points: 240 limbs have eight points per thread in the row pass, 255 and 320 sixteen where a prime is not just below 2^60)
@pytest.mark.parametrize("bits,mixed", [(50, False), (61, False), (60, True)])
def test_large_batches(bits, mixed):
    import torch
    log_n, pkg = 15, load_package()
    for polys, limbs in ((15, 16), (15, 17), (16, 20)):
        qs = pkg.primes_below(bits, log_n, limbs)
        if mixed:
            qs[-1] = around_the_line(log_n)[1]
        ctx = pkg.Context(log_n, qs, [], 1)
        q = torch.tensor(qs, dtype=torch.int64, device="cuda").view(-1, 1)
        gen = torch.Generator(device="cuda").manual_seed(limbs)
        a = torch.randint(0, 1 << 62, (polys, limbs, 1 << log_n), dtype=torch.int64, device="cuda", generator=gen).remainder_(q)
        a[0] = q - 1
        want = torch.cat([ctx.ntt(part.clone(), list(range(limbs))) for part in a.split(1)])   # four points: few limbs
        assert torch.equal(ctx.ntt(a, list(range(limbs))), want), limbs


@pytest.mark.parametrize("log_n", [10, 13, 16])
@pytest.mark.parametrize("largest", [False, True])
def test_key_switches_and_conversions(log_n, largest):
    """Chain and special primes of either kind: key products between the passes of their transforms, conversions from and to both kinds, and
    the tail of a ModDown."""
    above, below, top = around_the_line(log_n)
    others = [p for p in O.primes_below(60, log_n, 4) if p not in (above, top)]
    small = O.primes_below(42, log_n, 1)
    qs, ps, dnum = [above, others[0]] + small + [below], [top, others[1]], 2
    orc, ctx = O.Oracle(log_n, qs, ps, dnum), load_package().Context(log_n, qs, ps, dnum)
    rng, n = np.random.default_rng(log_n + 100 * largest), 1 << log_n
    key = residues(rng, qs + ps, (dnum, 2), n, largest)
    for nq in (4, 2):
        p = residues(rng, qs[:nq], (), n, largest)
        ob, oa = np.empty((nq, n), dtype=np.uint64), np.empty((nq, n), dtype=np.uint64)
        orc.L.orc_keyswitch(orc.h, O._p(p), O._p(key), nq, O._p(ob), O._p(oa))
        assert np.array_equal(host(ctx.keyswitch(dev(p), dev(key), nq)), np.stack([ob, oa])), nq
        for polys in (2, 16):
            y = residues(rng, qs[:nq] + ps, (polys,), n, largest)
            for drop in (False, True):
                assert np.array_equal(host(ctx.moddown_batch(dev(y), nq, drop)), orc.moddown_drop(y, nq, drop)), (nq, polys, drop)


@pytest.mark.parametrize("digits", [1, 2, 3])
@pytest.mark.parametrize("largest", [False, True])
def test_hoisted_sums(digits, largest):
    """One source, two masked ones under one key (whole masks and run tables), and a sum longer than the accumulators' corrections are apart."""
    log_n, shift, n = 10, 3, 1 << 10
    above, below, top = around_the_line(log_n)
    qs, ps, nq = [above, below, O.primes_below(60, log_n, 5)[4]][:digits], [top, O.primes_below(60, log_n, 5)[3]], digits
    orc, ctx = O.Oracle(log_n, qs, ps, digits), load_package().Context(log_n, qs, ps, digits)
    rng, primes = np.random.default_rng(digits), qs + ps
    ext, b = [residues(rng, primes, (digits,), n, largest) for _ in range(2)], [residues(rng, qs, (), n, largest) for _ in range(2)]
    keys = [residues(rng, primes, (digits, 2), n, largest) for _ in range(2)]
    full = [residues(rng, primes, (), n, largest) for _ in range(2)]
    runs = [np.repeat(residues(rng, primes, (), n >> shift, largest), 1 << shift, axis=-1) for _ in range(2)]
    g = [pow(5, 77, 2 * n), pow(5, 3, 2 * n)]
    sums = [[(0, 0, None, 0)], [(0, 0, full[0], 0), (1, 0, full[1], 0)], [(0, 0, runs[0], 0), (1, 0, runs[1], 0)],
            [(i & 1, i >> 1 & 1, full[i & 1], i >> 1 & 1) for i in range(20)]]
    d_ext, d_b, d_keys, d_full = [[dev(x) for x in v] for v in (ext, b, keys, full)]
    d_runs = [ctx.compact_mask(dev(m), shift) for m in runs]
    groups, want = [], np.zeros((len(sums), 2, nq + 2, n), dtype=np.uint64)
    for o, terms in enumerate(sums):
        group = []
        for i, (s, k, m, a) in enumerate(terms):
            table = o == 2
            mask = None if m is None else d_runs[s] if table else d_full[s]
            group.append((d_ext[s], d_b[s], d_keys[k], mask, g[a], shift) if table else (d_ext[s], d_b[s], d_keys[k], mask, g[a]))
            orc.L.orc_hoisted_term(orc.h, O._p(ext[s]), O._p(b[s]), O._p(keys[k]), O._p(m) if m is not None else None, g[a], nq, O._p(want[o]), int(i > 0))
        groups.append(group)
    for o, got in enumerate(host(ctx.hoisted_terms(groups, nq))):
        assert np.array_equal(got, want[o]), o
