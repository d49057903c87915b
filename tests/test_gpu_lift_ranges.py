"""Encodings whose coefficients lie on both sides of what a transform takes without reducing it (magnitudes of 2^51 for primes of 44 bits, of
the prime itself for larger ones), within a polynomial and from one thread's coefficients to the next: residues as the oracle's."""
import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log_n", [10, 12, 13, 16])
@pytest.mark.parametrize("top", [46, 51, 53])
def test_coefficients_around_the_ranges(log_n, top):
    import torch
    pkg = load_package()
    mods = [O.primes_below(60, log_n, 1)[0], O.primes_below(46, log_n, 1)[0], O.primes_below(44, log_n, 1)[0]]
    ctx, orc = pkg.Context(log_n, mods, [], 1), O.Oracle(log_n, mods, [], 1, threads=8)
    rng = np.random.default_rng(top)
    z = rng.normal(size=orc.slots) + 1j * rng.normal(size=orc.slots)
    scale = 2.0 ** top * np.sqrt(orc.slots)      # coefficients of about 2^top
    want = orc.encode(z, 2, scale)
    assert np.array_equal(ctx.encode(torch.from_numpy(z).cuda().reshape(1, -1), scale, 3).cpu().numpy().view(np.uint64)[0], want.data)
