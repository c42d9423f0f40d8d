"""Panel leaves of sgetrf at the edges of their shapes: one wave, several waves, one or two rows
per lane (64 / 128 / 256 / 512 / 1024 rows), several workgroups (1025, 8192 / 8193 rows), blocks
of eight columns, 32-column chunks and leaf widths with remainders. ipiv equals the oracle's
(LAPACK pivoting, lowest row on ties) and the backward error stays within 10 n eps."""
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


def _getrf(a, lda, pivot=True):
    import torch

    L = A.lib()
    m, n = a.shape
    d = A.to_device_cm(a, lda)
    lw = ctypes.c_int(0)
    with A.Handle() as h:
        assert L.aclsolverSgetrf_bufferSize(h.h, m, n, A.ptr(d), lda, ctypes.byref(lw)) == A.SUCCESS
        work = torch.empty(lw.value, device="cuda")
        ipiv = torch.zeros(min(m, n), dtype=torch.int32, device="cuda")
        info = torch.full((1,), -7, dtype=torch.int32, device="cuda")
        st = L.aclsolverSgetrf(h.h, m, n, A.ptr(d), lda, A.ptr(work), A.ptr(ipiv) if pivot else None, A.ptr(info))
        assert st == A.SUCCESS
        torch.cuda.synchronize()
    return A.from_device_cm(d, m, n), ipiv.cpu().numpy(), int(info.item())


@pytest.mark.parametrize("m", [1, 31, 63, 64, 65, 128, 129, 256, 257, 512, 513, 1024, 1025, 1280, 8192, 8193])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 31, 33, 57, 64, 65, 100])
def test_leaf_edges(m, n):
    print(f"leaf m={m} n={n}", flush=True)
    rng = np.random.default_rng(m * 131 + n)
    a = (rng.standard_normal((m, n)) / np.sqrt(min(m, n))).astype(np.float32)
    k = min(m, n)
    a[rng.permutation(m)[:k], np.arange(k)] += 2.0  # every column interchanges; no near ties
    lu, piv, info = _getrf(a, m + (n % 3))
    _, ref_piv, ref_info = O.sgetrf(a)
    assert info == ref_info == 0
    assert np.array_equal(piv, ref_piv)
    assert O.lu_backward_error(a, lu, piv) <= 10 * max(m, n) * EPS


@pytest.mark.parametrize("m,n", [(64, 64), (200, 70), (700, 64), (1500, 130)])
def test_leaf_ties_zero_columns_and_no_pivoting(m, n):
    """Entries of +-1 and 0 tie in every first column (lowest row wins), an exactly zero column
    gives info and leaves its rows as they are; without ipiv the diagonal is the pivot."""
    print(f"leaf ties m={m} n={n}", flush=True)
    rng = np.random.default_rng(m + n)
    a = np.zeros((m, n), np.float32)
    a[:, 0] = rng.choice([-1.0, 1.0], m)
    a[:, 1:] = rng.integers(-2, 3, (m, n - 1))
    a[:, 5] = 0.0
    lu, piv, info = _getrf(a, m)
    _, ref_piv, ref_info = O.sgetrf(a)
    assert ref_info == 6 and info == 6
    assert piv[0] == 1 and np.array_equal(piv[:6], ref_piv[:6])
    b = (rng.standard_normal((m, n)) / np.sqrt(n)).astype(np.float32)
    b[np.arange(n), np.arange(n)] += 4.0
    lu, _, info = _getrf(b, m, pivot=False)
    assert info == 0
    assert O.lu_backward_error(b, lu, np.arange(1, n + 1, dtype=np.int32)) <= 10 * m * EPS
