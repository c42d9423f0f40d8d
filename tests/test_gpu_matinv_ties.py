"""Batched inverses of orders 17..32 (two rows per lane, pivots by 32-bit maxima): pivots equal the
oracle's where magnitudes tie within a lane, between lanes and between the four matrices of a wave."""
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
EPS = 2.0 ** -24


@pytest.mark.parametrize("n", [17, 18, 24, 31, 32])
@pytest.mark.parametrize("batch", [1, 3, 18])
def test_ties(n, batch):
    """Small integers keep the first steps exact, so ties stay ties; |A C - I| within n eps |A| |C|
    (times 8) in the Frobenius norm."""
    import torch

    rng = np.random.default_rng(n * 100 + batch)
    mats = rng.integers(-1, 2, size=(batch, n, n)).astype(np.float32)
    mats[:, :, 0] = rng.choice([-1.0, 1.0], size=(batch, n))
    mats += (4 * n * np.eye(n, k=1) + 4 * n * np.eye(n, k=1 - n)).astype(np.float32)  # regular
    mats[:, n - 1, 0] = 1
    d = torch.from_numpy(np.ascontiguousarray(mats.transpose(0, 2, 1))).cuda()
    c = torch.zeros_like(d)
    ipiv = torch.zeros(batch * n, dtype=torch.int32, device="cuda")
    info = torch.full((batch,), -9, dtype=torch.int32, device="cuda")
    with A.Handle() as h:
        st = A.lib().aclsolverSmatinvStridedBatched(h.h, n, A.ptr(d), n, n * n, A.ptr(c), n, n * n, A.ptr(ipiv),
                                                    A.ptr(info), batch)
        torch.cuda.synchronize()
    assert st == A.SUCCESS
    got, piv = c.cpu().numpy().transpose(0, 2, 1), ipiv.cpu().numpy().reshape(batch, n)
    for i in range(batch):
        _, ref, ref_info, margin = O.sgetrf(mats[i], margins=True)
        assert int(info[i]) == ref_info == 0
        close = np.nonzero((margin < 1e-4) & (margin > 0))[0]  # near ties may turn with the rounding
        upto = int(close[0]) if len(close) else n
        assert piv[i][0] == 1 and np.array_equal(piv[i][:min(upto, 2)], ref[:min(upto, 2)])
        r = mats[i].astype(np.float64) @ got[i] - np.eye(n)
        assert np.linalg.norm(r) <= 8 * n * EPS * np.linalg.norm(mats[i]) * np.linalg.norm(got[i])
