"""Cross-workgroup waits that run out (a poll budget of zero, set from the host, so that every
kernel still exits): the interchange lists stay in range whatever the workspace held before, and
memory around the arguments is left alone."""
import contextlib
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

pytestmark = pytest.mark.gpu
POISON = 0x7F7F7F7F  # as a row index far beyond any matrix


@pytest.fixture(scope="module")
def handle():
    h = A.Handle()
    yield h
    h.close()


@contextlib.contextmanager
def no_polls():
    assert A.lib().aclsolverDebugSetSpinLimit(0) == A.SUCCESS
    try:
        yield
    finally:
        A.lib().aclsolverDebugSetSpinLimit(A.DEFAULT_SPIN_LIMIT)


@pytest.mark.parametrize("cplx,m,n", [(0, 1100, 1100), (0, 2304, 600), (0, 9000, 64), (1, 600, 600), (1, 9000, 64)])
def test_factorization_with_a_poisoned_workspace(handle, cplx, m, n):
    import torch

    print(f"timeout cplx={cplx} m={m} n={n}", flush=True)
    L, lda, guard = A.lib(), m + 5, 3
    dt = torch.complex64 if cplx else torch.float32
    a = torch.randn(n + guard, lda, dtype=dt, device="cuda")
    before = a.clone()
    lw = ctypes.c_int(0)
    size, getrf = (L.aclsolverCgetrf_bufferSize, L.aclsolverCgetrf) if cplx else (L.aclsolverSgetrf_bufferSize, L.aclsolverSgetrf)
    assert size(handle.h, m, n, A.ptr(a), lda, ctypes.byref(lw)) == A.SUCCESS
    words = lw.value * (2 if cplx else 1)
    work = torch.full((words + 4096,), POISON, dtype=torch.int32, device="cuda")
    ipiv = torch.full((min(m, n),), POISON, dtype=torch.int32, device="cuda")
    info = torch.full((1,), 7, dtype=torch.int32, device="cuda")
    with no_polls():
        assert getrf(handle.h, m, n, A.ptr(a), lda, A.ptr(work), A.ptr(ipiv), A.ptr(info)) == A.SUCCESS
        torch.cuda.synchronize()
    assert info.item() == A.INFO_WAIT_TIMEOUT
    piv = ipiv.cpu().numpy()
    assert np.all((piv >= 1) & (piv <= m))
    assert torch.isnan(torch.view_as_real(a[:64, :m]) if cplx else a[:64, :m]).all()
    assert torch.equal(a[n:], before[n:]) and torch.equal(a[:, m:], before[:, m:])
    assert bool((work[words:] == POISON).all())


@pytest.mark.parametrize("cplx", [0, 1])
@pytest.mark.parametrize("trans", [0, 1])
def test_host_solve_reports_the_wait(handle, cplx, trans):
    """Three blocks of 64 rows, so that a block waits for another; info stays as it was, as after
    any failed step of the staging."""
    print(f"host getrs cplx={cplx} trans={trans}", flush=True)
    n = 150
    a = np.eye(n, dtype=np.complex64 if cplx else np.float32) * 2
    a[1:, 0] = 0.5
    b = np.ones((n, 2), a.dtype)
    piv = np.arange(1, n + 1, dtype=np.int32)
    info = np.full(1, 7, np.int32)
    getrs = A.lib().aclsolverCgetrs if cplx else A.lib().aclsolverSgetrs

    def call():
        return getrs(handle.h, trans, n, 2, a.ctypes.data, n, piv.ctypes.data, b.ctypes.data, 2, info.ctypes.data)

    with no_polls():
        assert call() != 0
    assert info[0] == 7
    b[:] = 1
    assert call() == 0 and info[0] == 0
    assert np.isfinite(b).all()


def _diagonal(n, cplx=False):
    """Factors of 2 I with a nonzero first column of L: every block of rows waits for the first."""
    a = np.eye(n, dtype=np.complex64 if cplx else np.float32) * 2
    a[1:, 0] = 0.5
    return a


def test_getri_reports_the_wait(handle):
    import torch

    n = 150
    lu = A.to_device_cm(_diagonal(n))
    lw = ctypes.c_int(0)
    assert A.lib().aclsolverSgetri_bufferSize(handle.h, n, A.ptr(lu), n, ctypes.byref(lw)) == A.SUCCESS
    work = torch.zeros(lw.value, device="cuda")
    info = torch.full((1,), 7, dtype=torch.int32, device="cuda")

    def call(a):
        st = A.lib().aclsolverSgetri(handle.h, n, A.ptr(a), n, None, A.ptr(work), lw.value, A.ptr(info))
        torch.cuda.synchronize()
        return st, info.item()

    with no_polls():
        a = lu.clone()
        assert call(a) == (A.SUCCESS, A.INFO_WAIT_TIMEOUT)
        assert torch.isnan(a).any()
    assert call(lu.clone()) == (A.SUCCESS, 0)
    singular = lu.clone()
    singular[99, 99] = 0  # the factors stay, as before
    before = singular.clone()
    assert call(singular) == (A.SUCCESS, 100) and torch.equal(singular, before)


@pytest.mark.parametrize("cplx,n", [(0, 600), (1, 150)])
def test_getri_batched_reports_the_wait(handle, cplx, n):
    import torch

    print(f"getri_batched cplx={cplx} n={n}", flush=True)
    a = torch.stack([A.to_device_cm(_diagonal(n, cplx))] * 3)
    a[1, 70, 70] = 0
    c = torch.zeros_like(a)
    pa, pc = (torch.tensor([t[k].data_ptr() for k in range(3)], dtype=torch.int64, device="cuda") for t in (a, c))
    info = torch.full((3,), 7, dtype=torch.int32, device="cuda")
    getri = A.lib().aclsolverCgetriBatched if cplx else A.lib().aclsolverSgetriBatched

    def call():
        st = getri(handle.h, n, A.ptr(pa), n, None, A.ptr(pc), n, A.ptr(info), 3)
        torch.cuda.synchronize()
        return st, info.tolist()

    with no_polls():
        assert call() == (A.SUCCESS, [A.INFO_WAIT_TIMEOUT] * 3)
    assert call() == (A.SUCCESS, [0, 71, 0])


@pytest.mark.parametrize("cplx", [0, 1])
@pytest.mark.parametrize("trans", [0, 1])
@pytest.mark.parametrize("nrhs", [1, 40])
def test_device_solve_reports_the_wait(handle, cplx, trans, nrhs):
    import torch

    print(f"device getrs cplx={cplx} trans={trans} nrhs={nrhs}", flush=True)
    n = 150
    lu = A.to_device_cm(_diagonal(n, cplx))
    info = torch.full((1,), 7, dtype=torch.int32, device="cuda")
    getrs = A.lib().aclsolverCgetrsDevice if cplx else A.lib().aclsolverSgetrsDevice

    def call():
        b = torch.ones(nrhs, n, dtype=lu.dtype, device="cuda")
        st = getrs(handle.h, trans, n, nrhs, A.ptr(lu), n, None, A.ptr(b), n, A.ptr(info))
        torch.cuda.synchronize()
        return st, info.item(), bool(torch.isnan(torch.view_as_real(b) if cplx else b).any())

    with no_polls():
        assert call() == (A.SUCCESS, A.INFO_WAIT_TIMEOUT, True)
    assert call() == (A.SUCCESS, 0, False)
