"""Calls that would read or write beyond a mask or a message on the host are refused."""
import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def H():
    load_package()
    from efla_amd import hellm
    qs, ps = O.ckks_chain(10, 8, 3)
    return hellm.HEMMer(10, qs, ps, dnum=3, min_bootstrap_level=0, seed=4)


def tile(rows, cols):
    return np.random.default_rng(rows * 100 + cols).uniform(-1, 1, (rows, cols))


def test_blocks_beyond_the_tile(H):
    a = H.encrypt2(tile(16, 16), tile(16, 16))
    for call in (H.repack_to_one_col, H.repack_to_multi_col, H.get_low_col_block, H.repack_to_one_row, H.repack_to_multi_row, H.get_low_row_block):
        call(a, 7)
        for block in (8, 1 << 20):
            with pytest.raises(ValueError, match="no such block"):
                call(a, block)


def test_low_rank_products_of_thinner_tiles(H):
    thin, a = H.encrypt2(tile(1, 1), tile(1, 1)), H.encrypt2(tile(16, 16), tile(16, 16))
    for x, y in ((thin, thin), (a, thin)):
        for call in (lambda: H.matmul_high_low(x, y, 0, 2), lambda: H.matmul_low_high(x, y, 0, 2), lambda: H.matmul_low_low(x, y, 0, 0, 2)):
            with pytest.raises(Exception):
                call()
    for call in (H.packed_matmul_pre, H.packed_matmul_pre_rev):
        with pytest.raises(ValueError, match="two rows and columns"):
            call(thin, 2)


def test_odd_polynomial_whose_quotient_is_a_constant(H):
    """Degree 8 by blocks of two: the last quotient has a constant term only, of which an odd polynomial takes nothing"""
    x = np.linspace(-1, 1, 256).reshape(16, 16)
    c = [0, 0.5, 0, -0.25, 0, 0.125, 0, 0.0625, 0.75]
    with np.errstate(all="ignore"):
        got = H.decrypt(H.eval_odd_polynomial(H.encrypt(x), c, 2, 3))
    assert np.abs(got - sum(c[i] * x ** i for i in (1, 3, 5, 7))).max() < 1e-6
