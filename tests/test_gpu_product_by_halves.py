"""Products of two single tiles whose other tile block takes half of the shifts (tiles of 128 rows): residues as the oracle's, right above and
below the levels the route needs; and with a left operand of unknown content, which keeps the other route."""
import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle import hemmer_ref as R
from oracle import oracle as O

pytestmark = pytest.mark.gpu
SEED, CHAIN, T = 13, 9, 2


@pytest.fixture(scope="module")
def ring():
    load_package()
    from efla_amd import hellm
    qs, ps = O.ckks_chain(16, CHAIN, 4)
    H = hellm.HEMMer(16, qs, ps, dnum=3, min_bootstrap_level=0, seed=SEED)
    orc = O.Oracle(16, qs, ps, dnum=3, threads=8)
    orc.gen_secret(SEED)
    orc.gen_mult_key(SEED)
    orc.gen_conj_key(SEED)
    orc.key_seed = SEED
    return H, orc


def as_oracle(orc, ct):
    return O.Ct(ct.residues(), orc.delta[ct.info()["level"]])


@pytest.mark.parametrize("la, lb", [(T + 6, T + 6), (T + 6, T + 5), (T + 5, T + 5), (T + 6, T + 4)])
def test_levels(ring, la, lb):
    H, orc = ring
    n = H.dim
    rng = np.random.default_rng(la * 16 + lb)
    A, B = rng.uniform(-1, 1, (n, n)), rng.uniform(-1, 1, (n, n))
    a, b = (H.level_down(H.encrypt(m), lvl) if lvl < CHAIN - 1 else H.encrypt(m) for m, lvl in ((A, la), (B, lb)))
    c = H.single_cc_matmul(a, b, T)
    want = R.mult_mat_mat_cc_packed_single(orc, as_oracle(orc, a), as_oracle(orc, b), T, n, n)
    assert c.info()["level"] == T and np.array_equal(c.residues(), want.data)
    assert np.abs(H.decrypt(c) - A @ B).max() < 2.0 ** -12
    assert np.abs(H.decrypt_slots(c)[n * n:]).max() < 2.0 ** -12
    H.set_schedule(True, batch=3)
    again = H.single_cc_matmul(a, b, T).residues()
    H.set_schedule(True)
    assert np.array_equal(again, want.data)


def test_unknown_left_operand(ring):
    H, orc = ring
    n = H.dim
    rng = np.random.default_rng(3)
    A, A2, B = (rng.uniform(-1, 1, (n, n)) for _ in range(3))
    z = np.concatenate([A.reshape(-1), A2.reshape(-1)]).astype(np.complex128)
    oa = orc.encrypt(orc.encode(z, CHAIN - 1), 77)
    a, b = H.upload(oa.data, n, n, n), H.encrypt(B)
    c = H.single_cc_matmul(a, b, T)
    want = R.mult_mat_mat_cc_packed(orc, oa, as_oracle(orc, b), T, n, n, single_tile=True)
    assert np.array_equal(c.residues(), want.data)
    assert np.abs(H.decrypt(c) - A @ B).max() < 2.0 ** -12
