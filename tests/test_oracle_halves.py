"""The product by halves on the oracle's small ring: both blocks' shares of the sum over the shifts, put together."""
import numpy as np
import pytest

from oracle import hemmer_ref as R
from oracle import oracle as O


@pytest.mark.parametrize("target, la, lb", [(1, 7, 7), (1, 7, 6), (0, 6, 5), (0, 7, 7)])
def test_product_by_halves_over_oracle(target, la, lb):
    n = 16
    qs, ps = O.ckks_chain(10, 8, 3)
    orc = O.Oracle(10, qs, ps, dnum=3)
    orc.gen_secret(5)
    orc.gen_mult_key(5)
    orc.gen_conj_key(5)
    orc.key_seed = 5
    rng = np.random.default_rng(la)
    A, B = rng.uniform(-0.1, 0.1, (n, n)), rng.uniform(-1, 1, (n, n))
    a, b = (orc.level_down(orc.encrypt(orc.encode(m.reshape(-1), 7), 20 + i), lvl) if lvl < 7 else orc.encrypt(orc.encode(m.reshape(-1), 7), 20 + i)
            for i, (m, lvl) in enumerate(((A, la), (B, lb))))
    c = R.mult_mat_mat_cc_packed_halves(orc, a, b, target, n, n)
    assert c.level == target and c.scale == orc.delta[target]
    z = orc.decrypt(c)
    assert np.abs(z[: n * n].real.reshape(n, n) - A @ B).max() < 2 ** -18
    assert np.abs(z[n * n:]).max() < 2 ** -18 and np.abs(z.imag).max() < 2 ** -18
