"""U12 of wide matrices: the block solve of K = m rows, K with a remainder of the 64-row blocks and
16-row tiles, for numbers of columns around its 16-column strips."""
import ctypes
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


@pytest.mark.parametrize("m", [1, 15, 64, 65, 81, 130, 300, 511, 512, 513])
@pytest.mark.parametrize("extra", [1, 15, 16, 17, 100])
def test_wide_factors(m, extra):
    """Backward error within 10 n eps, pivots those of the oracle (no near ties by construction)."""
    import torch

    rng = np.random.default_rng(m * 1000 + extra)
    n, lda = m + extra, m + extra % 3
    a = (rng.standard_normal((m, n)) / np.sqrt(m)).astype(np.float32)
    a[rng.permutation(m), np.arange(m)] += 2.0
    L = A.lib()
    d = A.to_device_cm(a, lda)
    lw = ctypes.c_int(0)
    with A.Handle() as h:
        assert L.aclsolverSgetrf_bufferSize(h.h, m, n, A.ptr(d), lda, ctypes.byref(lw)) == A.SUCCESS
        work = torch.empty(lw.value, device="cuda")
        ipiv = torch.zeros(m, dtype=torch.int32, device="cuda")
        info = torch.full((1,), -7, dtype=torch.int32, device="cuda")
        assert L.aclsolverSgetrf(h.h, m, n, A.ptr(d), lda, A.ptr(work), A.ptr(ipiv), A.ptr(info)) == A.SUCCESS
        torch.cuda.synchronize()
    lu, piv = A.from_device_cm(d, m, n), ipiv.cpu().numpy()
    assert int(info.item()) == 0
    assert np.array_equal(piv, O.sgetrf(a)[1])
    assert O.lu_backward_error(a, lu, piv) <= 10 * n * EPS
