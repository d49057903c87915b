"""Basis conversions inside the first pass of a transform, against the oracle: every number of source limbs has code of its own, and
the sums are finished differently for primes below 2^44, of 59 or 60 bits and between."""
import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int64)).cuda()


def host(t):
    return t.cpu().numpy().view(np.uint64)


# the smallest primes a context takes (2^31 ...), both sides of 2^44, of 2^59, and the largest a conversion takes
TARGET_BITS = (32, 44, 45, 52, 59, 60)


@pytest.mark.parametrize("log_n", [11, 13, 16])   # one launch, two, and the pass whose rows are a compile-time constant
@pytest.mark.parametrize("n_src", range(1, 9))
def test_every_number_of_sources(log_n, n_src):
    """Two digits of n_src limbs, of 60 bits and of mixed sizes, to each other's primes and to special primes of every size; the first
    half of the coefficients of every scaled source residue is q - 1, the largest sums there are."""
    pkg = load_package()
    N = 1 << log_n
    big = pkg.primes_below(60, log_n, 2 * n_src + 1)
    ps = [pkg.primes_below(b, log_n, 1)[0] for b in TARGET_BITS[:-1]] + big[n_src:n_src + 1]
    sizes = [60, 50, 43, 57, 40, 59, 46, 55][:n_src]
    mixed = [big[n_src + 1 + i] if b == 60 else pkg.primes_below(b, log_n, 2)[1] for i, b in enumerate(sizes)]
    qs = big[:n_src] + mixed
    orc, ctx = O.Oracle(log_n, qs, ps, 2, threads=8), pkg.Context(log_n, qs, ps, 2)
    rng = np.random.default_rng(100 * log_n + n_src)
    poly = np.empty((2 * n_src, N), dtype=np.uint64)
    for j, q in enumerate(qs):
        basis = qs[:n_src] if j < n_src else qs[n_src:]
        hat = 1
        for r in basis:
            hat = hat * (r % q) % q if r != q else hat
        c = rng.integers(0, q, N, dtype=np.uint64)
        c[: N // 2] = (-hat) % q            # scaled by (S / q)^-1: q - 1
        poly[j] = c
    orc.ntt(poly, list(range(2 * n_src)))
    assert np.array_equal(host(ctx.modup_batch(dev(poly[None]), 2 * n_src)[0]), orc.modup(poly))
