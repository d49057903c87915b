"""Plaintext products over the diagonals of the weight, residue for residue against the oracle: rings whose table runs are wider and
narrower than a wavefront's residues, tiles that fill their rows and that do not, the lowest and other target levels, operands right above
the lowest level and at the top; and the products that stay with the shifts."""
import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle import hemmer_ref as R
from oracle import oracle as O

pytestmark = pytest.mark.gpu
SEED = 11


@pytest.fixture(scope="module")
def rings():
    load_package()
    from efla_amd import hellm
    made = {}

    def of(log_n):
        if log_n not in made:
            qs, ps = O.ckks_chain(log_n, 8, 3)
            orc = O.Oracle(log_n, qs, ps, dnum=3)
            orc.gen_secret(SEED)
            orc.gen_mult_key(SEED)
            orc.gen_conj_key(SEED)
            orc.key_seed = SEED
            made[log_n] = hellm.HEMMer(log_n, qs, ps, dnum=3, min_bootstrap_level=0, seed=SEED), orc
        return made[log_n]
    return of


def lowered(H, orc, ct, level):
    ct = H.level_down(ct, level) if ct.info()["level"] > level else ct
    return ct, O.Ct(ct.residues(), orc.delta[level])


@pytest.mark.parametrize("log_n, k, pair, level, target", [
    (10, 16, False, 7, 2), (10, 16, True, 4, 0), (10, 16, True, 7, 4), (10, 8, False, 5, 1), (10, 4, False, 7, 2),
    (12, 32, False, 6, 3), (12, 32, True, 5, 2), (12, 32, True, 7, 0), (14, 64, False, 4, 1), (14, 64, True, 7, 2)])
def test_product_over_the_diagonals(rings, log_n, k, pair, level, target):
    H, orc = rings(log_n)
    rng = np.random.default_rng(log_n * 100 + k + pair)
    A, A2, B, B2 = (rng.uniform(-1, 1, (k, k)) for _ in range(4))
    ct, want = lowered(H, orc, H.encrypt2(A, A2) if pair else H.encrypt(A), level)
    pt = H.encode2(B, B2) if pair else H.encode(B)
    w = ct.info()["block_width"]
    got = H.single_matmul(ct, pt, target)
    want = R.mult_mat_mat_pc_lazy(orc, want, O.Pt(pt.residues(), orc.delta[orc.nQ - 1]), target, k, w)
    assert got.info()["level"] == target
    assert np.array_equal(got.residues(), want.data)
    if target > 0:    # (at level 0 the products may pass the first prime's half)
        d = H.decrypt2(got) if pair else [H.decrypt(got)]
        for c, x in zip(d, [A @ B, A2 @ B2]):
            assert np.abs(c - x).max() < 2.0 ** -14
    assert np.array_equal(H.single_matmul(ct, pt, target).residues(), got.residues())


def test_unknown_left_operand_of_a_single_tile_keeps_its_masks(rings):
    """The diagonals of a single tile act on every block alike: an operand that may carry something in its other blocks takes the
    shifts, whose masks keep the product empty there."""
    H, orc = rings(10)
    rng = np.random.default_rng(5)
    z = rng.uniform(-1, 1, orc.slots).astype(np.complex128)
    B = rng.uniform(-1, 1, (16, 16))
    a = orc.encrypt(orc.encode(z, 7), 1234)
    ct = H.upload(a.data, 16, 16, 16)
    pt = H.encode(B)
    got = H.single_matmul(ct, pt, 2)
    want = R.mult_mat_mat_pc_lazy(orc, a, O.Pt(pt.residues(), orc.delta[7]), 2, 16, 16, a_known=False)
    assert np.array_equal(got.residues(), want.data)
    s = H.decrypt_slots(got)
    assert np.abs(s[:256].real.reshape(16, 16) - z[:256].real.reshape(16, 16) @ B).max() < 2.0 ** -18
    assert np.abs(s[256:]).max() < 2.0 ** -20


@pytest.mark.parametrize("a_level, b_level", [(6, 7), (7, 3)])   # A not three levels above the target; B below what the products ask for
def test_a_refused_product_derives_no_keys(rings, a_level, b_level):
    from efla_amd import hellm
    _, orc = rings(10)
    H = hellm.HEMMer(10, orc.q, orc.p, dnum=3, min_bootstrap_level=3, seed=SEED)
    rng = np.random.default_rng(3)
    A, B = rng.uniform(-1, 1, (16, 16)), rng.uniform(-1, 1, (16, 16))
    ct = H.encrypt(A)
    ct, pt = H.level_down(ct, a_level) if a_level < 7 else ct, H.encode(B, b_level)
    held = H.key_bytes()
    with pytest.raises(Exception, match="level >= "):
        H.single_matmul(ct, pt, 4)
    after = H.key_bytes()
    assert (after["plain"], after["compact"]) == (held["plain"], held["compact"])
    assert np.abs(H.decrypt(H.single_matmul(H.encrypt(A), H.encode(B), 4)) - A @ B).max() < 2.0 ** -14
    assert H.key_bytes()["compact"] > held["compact"]


def test_a_weight_is_decoded_once(rings):
    """What a product with a new weight takes more than one with a known weight: its decoding, and one transform where tau(B) is encoded
    (the diagonals' tables are made without one)."""
    H, orc = rings(10)
    rng = np.random.default_rng(8)
    A = H.encrypt(rng.uniform(-1, 1, (16, 16)))
    unknown = H.upload(A.residues(), 16, 16, 16)

    def transforms(a, w):
        H.traffic(reset=True)
        H.single_matmul(a, w, 2)
        return H.traffic(reset=True)[1]["transforms"]

    for a, more in ((A, 1), (unknown, 2)):
        first, second = (H.encode(rng.uniform(-1, 1, (16, 16))) for _ in range(2))
        transforms(a, first)
        known = transforms(a, first)
        assert transforms(a, second) == known + more
        assert transforms(a, second) == known


def test_tables_are_bounded_by_their_bytes():
    """Weights on the preset at target level 9, 31.5 MB of tables each: no more than 6 GiB of them are held, and the oldest is prepared again."""
    load_package()
    from efla_amd import hellm
    H = hellm.HEMMer(preset=True, seed=SEED)
    rng = np.random.default_rng(2)
    B = rng.uniform(-1, 1, (128, 128))
    a = H.encrypt2(B, B)
    tables = 15 * 512 * 32 * 8 * 16
    room = 6 * 1024 ** 3 // tables

    def transforms(i):   # of the product with weight i
        w = H.encode2(np.roll(B, i % 128, 1), np.roll(B, i // 128, 0), 10)
        H.traffic(reset=True)
        H.single_matmul(a, w, 9)
        return H.traffic(reset=True)[1]["transforms"]

    transforms(0)
    known = transforms(0)
    held = H.key_bytes()["pool"]
    for i in range(1, room + 24):
        assert transforms(i) == known + 2   # (decoding it is two launches)
    grown = H.key_bytes()["pool"] - held
    assert (room - 2) * tables < grown < 6 * 1024 ** 3
    assert transforms(room + 23) == transforms(24) == known
    assert transforms(23) == known + 2
