"""Chains whose results lie in buffers of their own (hemm_hoisted_moddown_to, hemm_rescale_to): the residues of the forms that leave
them back to back, which other tests compare with the oracle; and what the ciphertexts of a batch hold on to."""
import ctypes

import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def residues(primes, lead, N, gen):
    import torch
    q = torch.tensor(primes, dtype=torch.int64, device="cuda").view(-1, 1)
    return torch.randint(0, 1 << 62, tuple(lead) + (len(primes), N), dtype=torch.int64, device="cuda", generator=gen).remainder_(q)


def apart(n, stride_words):
    """n buffers for two polynomials each, in no order, with a guard word behind each polynomial"""
    import torch
    room = torch.full((n, 2 * stride_words), -1, dtype=torch.int64, device="cuda")
    order = [(7 * i + 3) % n if n % 7 else n - 1 - i for i in range(n)]
    bufs = [room[o] for o in order]
    return bufs, (ctypes.c_void_p * n)(*[b.data_ptr() for b in bufs])


# rings of every form of the tail: none (2^9), one launch (2^10 - 2^12, and 2^13 from 64 limbs), two launches; more results than a
# list holds; a conversion too wide to be fused, whose transform is cut into runs that start at an odd polynomial (2^16, 9 + 9)
@pytest.mark.parametrize("log_n,chain,special,n_out", [(9, 4, 2, 3), (10, 4, 2, 1), (11, 5, 2, 33), (12, 5, 2, 3), (13, 5, 2, 2),
                                                       (13, 5, 2, 9), (14, 6, 2, 5), (15, 4, 1, 3), (16, 4, 2, 1), (16, 7, 4, 5),
                                                       (16, 9, 9, 32)])
@pytest.mark.parametrize("drop", [0, 1])
def test_hoisted_moddown_to(log_n, chain, special, n_out, drop):
    import torch
    pkg = load_package()
    qs, ps = O.ckks_chain(log_n, chain, special)
    ctx, N, nq = pkg.Context(log_n, qs, ps, 1), 1 << log_n, chain
    gen = torch.Generator(device="cuda").manual_seed(log_n * 100 + n_out)
    ext, b, key = residues(qs + ps, (2, 1), N, gen), residues(qs, (2,), N, gen), residues(qs + ps, (1, 2), N, gen)
    groups = [[(ext[o % 2], b[(o + 1) % 2], key, None, pow(5, o, 2 * N))] for o in range(n_out)]
    want = ctx.hoisted_moddown(groups, nq, drop)
    nq_out = nq - drop
    stride = nq_out * N + 2
    bufs, outs = apart(n_out, stride)
    arr = (pkg.RotTerm * n_out)()
    for o, ((e, bb, k, _, g),) in enumerate(groups):
        arr[o] = pkg.RotTerm(e.data_ptr(), bb.data_ptr(), k.data_ptr(), None, g, 0, None, 1, 0)
    off = (ctypes.c_uint32 * (n_out + 1))(*range(n_out + 1))
    y = torch.empty((n_out, 2, nq + special, N), dtype=torch.int64, device="cuda")
    ws = torch.empty((n_out, 2, nq_out, N), dtype=torch.int64, device="cuda")
    pkg.check(pkg.lib().hemm_hoisted_moddown_to(ctx.h, arr, off, n_out, nq, 0, drop, y.data_ptr(), outs, stride, ws.data_ptr(), None))
    for o in range(n_out):
        got = bufs[o].view(2, stride)
        assert torch.equal(got[:, : nq_out * N].reshape(2, nq_out, N), want[o]), o
        assert bool((got[:, nq_out * N:] == -1).all()), o


@pytest.mark.parametrize("log_n,chain,n_out", [(9, 3, 2), (10, 4, 1), (11, 2, 33), (13, 4, 3), (13, 6, 8), (16, 2, 3), (16, 7, 4)])
def test_rescale_to(log_n, chain, n_out):
    import torch
    pkg = load_package()
    qs, ps = O.ckks_chain(log_n, 10, 4)   # scratch for 140 limbs
    ctx, N, nq = pkg.Context(log_n, qs, ps, 3), 1 << log_n, chain
    gen = torch.Generator(device="cuda").manual_seed(log_n + n_out)
    x = residues(qs[:nq], (n_out, 2), N, gen)
    want = torch.stack([ctx.rescale(x[o].contiguous(), nq) for o in range(n_out)])
    stride = (nq - 1) * N + 2
    bufs, outs = apart(n_out, stride)
    keep = x.clone()
    pkg.check(pkg.lib().hemm_rescale_to(ctx.h, x.data_ptr(), nq * N, outs, stride, nq, n_out, None))
    for o in range(n_out):
        got = bufs[o].view(2, stride)
        assert torch.equal(got[:, : (nq - 1) * N].reshape(2, nq - 1, N), want[o]), o
        assert bool((got[:, (nq - 1) * N:] == -1).all()), o
    assert torch.equal(x, keep)


def test_result_lists_are_checked():
    import torch
    pkg = load_package()
    qs, ps = O.ckks_chain(10, 4, 2)
    ctx, N, nq = pkg.Context(10, qs, ps, 3), 1 << 10, 4
    x = torch.zeros((2, 2, nq, N), dtype=torch.int64, device="cuda")
    r = torch.zeros((2, 2, nq - 1, N), dtype=torch.int64, device="cuda")

    def call(outs, in_stride=nq * N, out_stride=(nq - 1) * N, n=2):
        return pkg.lib().hemm_rescale_to(ctx.h, x.data_ptr(), in_stride, (ctypes.c_void_p * n)(*outs), out_stride, nq, n, None)

    a, b = r[0].data_ptr(), r[1].data_ptr()
    assert call([a, b]) == 0
    assert call([a, None]) == 1
    assert call([a, x[1].data_ptr()]) == 1                  # a result over an input
    assert call([a, x.data_ptr() - 8 * (2 * (nq - 1) * N - 1)]) == 1   # by one word
    assert call([a, b], in_stride=nq * N - 1) == 1
    assert call([a, b], out_stride=(nq - 1) * N - 1) == 1
    assert pkg.lib().hemm_rescale_to(ctx.h, x.data_ptr(), nq * N, None, (nq - 1) * N, nq, 2, None) == 1
    torch.cuda.synchronize()


def test_one_of_two_results_keeps_only_its_own_memory():
    """Two results of one batched call, one of them dropped: what the kept ones hold is theirs alone."""
    import torch
    pkg = load_package()
    from efla_amd import hellm
    qs, ps = O.ckks_chain(14, 9, 4)
    H = hellm.HEMMer(14, qs, ps, dnum=3, min_bootstrap_level=0, seed=5)
    rng = np.random.default_rng(1)
    m = rng.normal(size=(H.dim, H.dim))
    x = H.encrypt2(m, m)
    kept, count = [], 48

    def once():
        a, b = x.clone(), x.clone()
        H.one_mat_rot_sum_inplace(a, b)
        return a

    for _ in range(2):   # keys, pools, the first allocations of the runtime
        kept.append(once())
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    for _ in range(count):
        kept.append(once())
    torch.cuda.synchronize()
    own = 2 * len(qs) * 8 << 14                  # a ciphertext
    taken = (free - torch.cuda.mem_get_info()[0]) / count
    assert taken < 1.5 * own, (taken, own)       # a shared buffer holds two; allocations are rounded up a little
    assert np.array_equal(kept[0].residues(), kept[-1].residues())


def test_shifts_on_two_streams_share_one_workspace():
    """The column shifts of an activation run in two chains side by side; their workspaces together are one for `batch` shifts."""
    import torch
    pkg = load_package()
    from efla_amd import hellm
    log_n, target, special = 14, 4, 4
    qs, ps = O.ckks_chain(log_n, 9, special)
    H = hellm.HEMMer(log_n, qs, ps, dnum=3, min_bootstrap_level=0, seed=5)
    x = H.encrypt(np.random.default_rng(1).normal(size=(H.dim, H.dim)))
    H.set_schedule(True, 4)
    a = H.matmul_pre(x, target)                  # keys, masks, and as many results as the call below takes from the pool
    first = a.get(H.dim - 1, H.dim, H.dim, H.dim).residues()
    a.free()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    H.set_schedule(True, 16)
    b = H.matmul_pre(x, target)
    torch.cuda.synchronize()
    taken = free - torch.cuda.mem_get_info()[0]
    nq = target + 3
    workspace = 16 * 2 * ((nq + special) + (nq - 1)) * 8 << log_n
    assert taken < 1.25 * workspace, (taken, workspace)
    assert np.array_equal(first, b.get(H.dim - 1, H.dim, H.dim, H.dim).residues())
