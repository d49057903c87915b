"""Passes of four, eight and sixteen points per thread: both sides of the lines between them, against the oracle."""
import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _context(log_n):
    pkg = load_package()
    mods = [O.primes_below(61, log_n, 1)[0], O.primes_below(60, log_n, 1)[0], O.primes_below(42, log_n, 1)[0]]
    return pkg.Context(log_n, mods, [], 1), O.Oracle(log_n, mods, [], 1, threads=8), mods


# limbs at which a pass changes: columns at 512 workgroups of 4096 points (of 2^16 points half slabs at 384), rows at 640 and (forward) 900,
# one-launch transforms at 256 limbs
@pytest.mark.parametrize("log_n,limbs", [(10, 2), (11, 2), (12, 1), (12, 256), (12, 257), (13, 1), (14, 81), (15, 64), (15, 65), (15, 80), (15, 81),
                                         (15, 112), (15, 113), (16, 1), (16, 24), (16, 25), (16, 32), (16, 33), (16, 40), (16, 41), (16, 56),
                                         (16, 57)])
def test_transforms(log_n, limbs):
    import torch
    ctx, orc, mods = _context(log_n)
    rng = np.random.default_rng(limbs)
    for prime, q in enumerate(mods):
        a = rng.integers(0, q, (limbs, 1, 1 << log_n), dtype=np.uint64)
        a[0] = q - 1
        d = torch.from_numpy(a.view(np.int64)).cuda()
        ctx.ntt(d, [prime])
        got = d.cpu().numpy().view(np.uint64)
        for p in {0, limbs // 2, limbs - 1}:
            want = a[p].copy()
            orc.ntt(want, [prime])
            assert np.array_equal(got[p], want), (prime, p)
        ctx.ntt(d, [prime], inverse=True)
        assert np.array_equal(d.cpu().numpy().view(np.uint64), a), prime


# conversions at 256 workgroups of 4096 points (2^16 points: at 768), the row passes behind them at 640 and 900: a rescale of `polys` polynomials
# of nq limbs launches polys (nq - 1) limbs
@pytest.mark.parametrize("log_n,polys,nq", [(11, 2, 4), (12, 2, 18), (13, 2, 4), (14, 4, 17), (14, 4, 18), (15, 2, 17), (15, 2, 18), (15, 5, 17),
                                            (15, 9, 10), (15, 7, 17), (15, 8, 16), (16, 2, 9), (16, 4, 11), (16, 3, 15), (16, 3, 17), (16, 3, 18),
                                            (16, 7, 9), (16, 6, 11)])
def test_conversions(log_n, polys, nq):
    import torch
    pkg = load_package()
    mods = O.primes_below(60, log_n, 9) + O.primes_below(42, log_n, 9)
    ctx, orc = pkg.Context(log_n, mods, [], 1), O.Oracle(log_n, mods, [], 1, threads=8)
    rng = np.random.default_rng(polys)
    a = np.stack([rng.integers(0, q, (polys, 1 << log_n), dtype=np.uint64) for q in mods[:nq]], axis=1)
    a[0, -1] = mods[nq - 1] - 1
    got = ctx.rescale(torch.from_numpy(a.view(np.int64)).cuda(), nq).cpu().numpy().view(np.uint64)
    assert np.array_equal(got, orc.rescale(O.Ct(a.copy(), 1.0)).data)


# lifts of encodings, three limbs a message: slabs at 128 and 512 workgroups of 4096 points (2^16 points: at 1024), points per thread at 256,
# the row passes behind them at 640 and 900 (2^14 points: at 512 and 640); 2^13 points take one launch from 64 limbs on
@pytest.mark.parametrize("log_n,messages", [(13, 1), (13, 21), (13, 22), (14, 10), (14, 11), (14, 21), (14, 22), (14, 42), (14, 43), (14, 53), (14, 54),
                                            (15, 5), (15, 6), (15, 10), (15, 11), (15, 21), (15, 22), (15, 26), (15, 27), (15, 37), (15, 38),
                                            (16, 1), (16, 13), (16, 14), (16, 18), (16, 19), (16, 21), (16, 22)])
def test_lifts(log_n, messages):
    import torch
    pkg = load_package()
    mods = O.primes_below(60, log_n, 1) + O.primes_below(42, log_n, 2)
    ctx, orc = pkg.Context(log_n, mods, [], 1), O.Oracle(log_n, mods, [], 1, threads=8)
    rng = np.random.default_rng(messages)
    z = rng.uniform(-1, 1, (messages, 1 << (log_n - 1))) + 1j * rng.uniform(-1, 1, (messages, 1 << (log_n - 1)))
    got = ctx.encode(torch.from_numpy(z).cuda(), float(2**40), 3).cpu().numpy().view(np.uint64)
    for p in {0, messages // 2, messages - 1}:
        assert np.array_equal(got[p], orc.encode(z[p], 2, 2.0**40).data), p
