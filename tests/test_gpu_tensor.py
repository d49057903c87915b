"""The tensor product of two ciphertexts against integers: primes below 2^44, just below 2^60, of 60 bits and less but further off, and of 61
bits; random operands and every one at q - 1."""
import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle import oracle as O

pytestmark = pytest.mark.gpu
LOG_N = 10
N = 1 << LOG_N


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int64)).cuda()


@pytest.mark.parametrize("largest", [False, True])
def test_tensor_product(largest):
    step = 2 << LOG_N
    far = next(p for p in range((2**60 - 2**27) // step * step + 1 - step, 0, -step) if O.is_prime(p))
    qs = O.primes_below(42, LOG_N, 1) + O.primes_below(44, LOG_N, 1) + O.primes_below(60, LOG_N, 1) + [far] + O.primes_below(50, LOG_N, 1)
    qs += [O.nearest_prime(2**61 - 2**20, LOG_N)]
    ctx, nq, rng = load_package().Context(LOG_N, qs, [], 1), len(qs), np.random.default_rng(17)
    mods = np.array(qs, dtype=object).reshape(-1, 1)

    def residues(*lead):
        if largest:
            return np.broadcast_to(np.array(qs, dtype=np.uint64).reshape(-1, 1) - np.uint64(1), lead + (nq, N)).copy()
        return np.stack([rng.integers(0, q, lead + (N,), dtype=np.uint64) for q in qs], axis=-2)

    x, y = residues(2), residues(2)
    (b1, a1), (b2, a2) = x.astype(object), y.astype(object)
    want = (np.stack([b1 * b2, a1 * b2 + a2 * b1, a1 * a2]) % mods).astype(np.uint64)
    assert np.array_equal(ctx.tensor(dev(x), dev(y), nq).cpu().numpy().view(np.uint64), want)
