"""Tied pivot candidates in the batched inverses: the lowest row wins at every step, over all orders
and layouts of the kernels (several matrices a wave, two rows a lane, a wave per matrix)."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for p in (ROOT, os.path.join(ROOT, "ops-solver_amd")):
    if p not in sys.path:
        sys.path.insert(0, p)

import aclsolver as A  # noqa: E402
from oracle import oracle as O  # noqa: E402

pytestmark = pytest.mark.gpu


def tied(rng, n):
    """L U with rows permuted, L's entries 0 or +-1 and U small integers over a diagonal of +-1: every
    step of an elimination has ties, exact ones."""
    lo = np.eye(n) + np.tril(rng.integers(-1, 2, (n, n)) * (rng.random((n, n)) < 0.3), -1)
    up = np.diag(rng.choice([-1.0, 1.0], n)) + np.triu(rng.integers(-1, 2, (n, n)) * (rng.random((n, n)) < 0.1), 1)
    return (lo @ up)[rng.permutation(n)].astype(np.float32)


@pytest.mark.parametrize("n", [7, 8, 13, 16, 17, 18, 25, 31, 32, 33, 64])
def test_real_pivots(n):
    """Pivots equal the oracle's up to the first step whose candidates nearly, but not exactly, tie
    (the rounding may turn those); the 24 matrices pin at least 50 tied steps."""
    import torch

    rng = np.random.default_rng(n)
    batch, pinned = 24, 0
    mats = np.stack([tied(rng, n) for _ in range(batch)])
    d = torch.from_numpy(np.ascontiguousarray(mats.transpose(0, 2, 1))).cuda()
    c = torch.zeros_like(d)
    ipiv = torch.zeros(batch * n, dtype=torch.int32, device="cuda")
    info = torch.full((batch,), -9, dtype=torch.int32, device="cuda")
    with A.Handle() as h:
        assert A.lib().aclsolverSmatinvStridedBatched(h.h, n, A.ptr(d), n, n * n, A.ptr(c), n, n * n, A.ptr(ipiv),
                                                      A.ptr(info), batch) == A.SUCCESS
        torch.cuda.synchronize()
    piv = ipiv.cpu().numpy().reshape(batch, n)
    for i in range(batch):
        _, ref, ref_info, margin = O.sgetrf(mats[i], margins=True)
        assert int(info[i]) == ref_info == 0
        near = np.nonzero((margin < 1e-4) & (margin > 0))[0]
        upto = int(near[0]) if len(near) else n
        pinned += int(np.sum(margin[:upto] == 0))
        assert np.array_equal(piv[i][:upto], ref[:upto])
    assert pinned >= 50


@pytest.mark.parametrize("n", [5, 8, 13, 16, 20, 32, 33, 40, 47, 63, 64])
@pytest.mark.parametrize("exact_first", [True, False])
def test_complex_choice(n, exact_first):
    """Two rows tie in the first column with 4 and 1 + 3j (largest |re| + |im| by far), and the second
    column is the first times a number of few bits. With the pivot 4 every multiplier and product is
    exact, so the second step finds only zeros: info = 2. With 1 + 3j the multipliers are rounded
    and remainders stay. So info tells which of the two rows was taken."""
    import torch

    rng = np.random.default_rng(n + exact_first)
    batch = 6
    a = np.zeros((batch, n, n), np.complex64)
    for i in range(batch):
        col = (rng.integers(-64, 65, n) + 1j * rng.integers(-64, 65, n)) / 64
        low, high = sorted(rng.choice(n, 2, replace=False))
        col[low], col[high] = (4, 1 + 3j) if exact_first else (1 + 3j, 4)
        a[i] = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
        a[i, :, 0] = col
        a[i, :, 1] = col * (3 + 5j)
    t = torch.from_numpy(np.ascontiguousarray(a.transpose(0, 2, 1))).cuda()
    c = torch.zeros_like(t)
    pa, pc = (torch.tensor([x[i].data_ptr() for i in range(batch)], dtype=torch.int64, device="cuda") for x in (t, c))
    info = torch.full((batch,), -9, dtype=torch.int32, device="cuda")
    with A.Handle() as h:
        assert A.lib().aclsolverCmatinvBatched(h.h, n, A.ptr(pa), n, A.ptr(pc), n, A.ptr(info), batch) == A.SUCCESS
        torch.cuda.synchronize()
    got = info.cpu().numpy()
    assert np.all(got == 2) if exact_first else np.all(got != 2)
