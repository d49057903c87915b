"""Matrices on their way to the GPU through pinned host memory."""
import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log_n", [10, 16])
def test_more_matrices_in_the_queue_than_pinned_stages(log_n):
    """Matrices that wait for the GPU in pinned memory: a ninth user of the eight stages waits for the first one's work."""
    import torch
    load_package()
    from efla_amd import hellm
    qs, ps = O.ckks_chain(log_n, 4, 2)
    H = hellm.HEMMer(log_n, qs, ps, dnum=2, min_bootstrap_level=0, seed=9)
    rng = np.random.default_rng(2)
    m = [rng.uniform(-1, 1, (H.dim, H.dim)) for _ in range(27)]
    H.decrypt(H.encrypt(m[0]))                   # tables, stages
    torch.cuda.synchronize()
    busy = torch.zeros(1 << 26, device="cuda")
    for _ in range(400):                         # work in front, so that nothing has been read when the ninth matrix comes
        busy.add_(1.0)
    ahead = torch.cuda.Event()
    ahead.record()
    cts, waiting = [], 0
    for i in range(0, 27, 3):                    # three stages each, one after the other
        cts.append((H.encrypt(m[i]), H.encrypt2(m[i + 1], m[i + 2]), H.encode(m[i])))
        waiting += not ahead.query()
    assert waiting >= 2                          # the queue was full when the ninth user came
    for (a, b, p), i in zip(cts, range(0, 27, 3)):
        assert np.abs(H.decrypt(a) - m[i]).max() < 1e-6
        assert all(np.abs(x - y).max() < 1e-6 for x, y in zip(H.decrypt2(b), m[i + 1:i + 3]))
        assert np.array_equal(p.residues(), H.encode(m[i]).residues())
