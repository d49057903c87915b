"""Column passes on slabs of a half and a quarter of the columns (rings of 2^13 to 2^15 points, few limbs): both sides of the lines, both
arithmetics and primes above 2^60, forward and back, against the oracle."""
import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle import oracle as O

pytestmark = pytest.mark.gpu


# limbs at which the slabs change: 2^13 at 64 (one launch from there), 2^14 at 32, 2^15 at 16 (forward) and 64
@pytest.mark.parametrize("log_n,polys", [(13, 1), (13, 21), (14, 1), (14, 10), (14, 11), (14, 31), (15, 1), (15, 5), (15, 6), (15, 21), (15, 22)])
def test_transforms_on_both_sides_of_the_lines(log_n, polys):
    import torch
    pkg = load_package()
    mods = [O.primes_below(61, log_n, 1)[0], O.primes_below(60, log_n, 1)[0], O.primes_below(42, log_n, 1)[0]]
    ctx, orc = pkg.Context(log_n, mods, [], 1), O.Oracle(log_n, mods, [], 1, threads=8)
    rng = np.random.default_rng(polys)
    a = np.stack([[rng.integers(0, q, 1 << log_n, dtype=np.uint64) for q in mods] for _ in range(polys)])
    d = torch.from_numpy(a.view(np.int64)).cuda()
    ctx.ntt(d, [0, 1, 2])
    got = d.cpu().numpy().view(np.uint64)
    for p in {0, polys // 2, polys - 1}:
        want = a[p].copy()
        orc.ntt(want, [0, 1, 2])
        assert np.array_equal(got[p], want), p
    ctx.ntt(d, [0, 1, 2], inverse=True)
    assert np.array_equal(d.cpu().numpy().view(np.uint64), a)
