"""Factorizations whose unit-lower blocks have large inverses (multipliers of one sign, or large
ones without pivoting), and rows that overflow: U comes as from a substitution."""
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
EPS = 2.0 ** -24
KINDS = [np.float32, np.complex64]


@pytest.fixture(scope="module")
def handle():
    h = A.Handle()
    yield h
    h.close()


def factor(handle, a, pivoting=True, tournament=False):
    import torch

    m, n = a.shape
    cplx, L = np.iscomplexobj(a), A.lib()
    print(f"factor {a.dtype} {m} x {n} pivoting={pivoting} tournament={tournament}", flush=True)
    size = L.aclsolverCgetrf_bufferSize if cplx else L.aclsolverSgetrf_bufferSize
    getrf = L.aclsolverCgetrf if cplx else (L.aclsolverSgetrfTournament if tournament else L.aclsolverSgetrf)
    d = A.to_device_cm(a)
    lw = ctypes.c_int(0)
    assert size(handle.h, m, n, A.ptr(d), m, ctypes.byref(lw)) == A.SUCCESS
    work = torch.empty(lw.value, dtype=d.dtype, device="cuda")
    ipiv = torch.zeros(min(m, n), dtype=torch.int32, device="cuda") if pivoting else None
    info = torch.full((1,), -7, dtype=torch.int32, device="cuda")
    assert getrf(handle.h, m, n, A.ptr(d), m, A.ptr(work), A.ptr(ipiv), A.ptr(info)) == A.SUCCESS
    torch.cuda.synchronize()
    assert info.item() == 0
    return A.from_device_cm(d, m, n), ipiv.cpu().numpy() if pivoting else None


def parts(lu):
    """L (unit lower) and U in 64-bit parts."""
    m, n = lu.shape
    k = min(m, n)
    wide = lu.astype(np.complex128 if np.iscomplexobj(lu) else np.float64)
    return np.tril(wide[:, :k], -1) + np.eye(m, k), np.triu(wide[:k])


def upper(rng, n, dtype):
    u = np.triu(rng.standard_normal((n, n)) + (1j * rng.standard_normal((n, n)) if dtype == np.complex64 else 0), 1)
    return u + np.diag(rng.uniform(1, 2, n))


@pytest.mark.parametrize("dtype", KINDS)
@pytest.mark.parametrize("c", [0.3, 0.5, 1.0])
@pytest.mark.parametrize("n", [65, 100, 128, 300, 700, 1300])
def test_multipliers_of_one_sign(handle, dtype, c, n):
    """A = L U with -c everywhere below L's diagonal. The bound on |P A - L U| is a substitution's,
    n eps |L| |U|, with the largest entry of the product and a factor of 10 for complex products
    and the growth of 16 columns."""
    rng = np.random.default_rng(n)
    a = ((np.eye(n) - c * np.tri(n, k=-1)) @ upper(rng, n, dtype)).astype(dtype)
    for tournament in (False, True) if dtype == np.float32 and n > 1024 else (False,):
        lu, piv = factor(handle, a, tournament=tournament)
        rows = np.arange(n)
        for j, r in enumerate(piv):
            rows[[j, r - 1]] = rows[[r - 1, j]]
        lo, up = parts(lu)
        assert np.abs(a[rows] - lo @ up).max() <= 10 * n * EPS * (np.abs(lo) @ np.abs(up)).max()


def exact_factors(rng, n, dtype):
    """L with about three entries of 2^17 a row and U of small integers, pivots powers of two: every
    number that an elimination meets has at most 21 bits, so that it gives exactly these factors,
    while inv(L) grows like 2^(17 k)."""
    unit = [1, -1, 1j, -1j] if dtype == np.complex64 else [1, -1]
    lo = np.eye(n, dtype=np.complex128 if dtype == np.complex64 else np.float64)
    for i in range(1, n):
        for j in {i - 1} | set(rng.integers(0, i, 2).tolist()):
            lo[i, j] = rng.choice(unit) * 2 ** 17
    up = np.triu(rng.integers(-2, 3, (n, n)), 1) + np.diag(rng.choice([1, -1, 2, -2], n))
    return lo, up.astype(lo.dtype)


@pytest.mark.parametrize("dtype", KINDS)
@pytest.mark.parametrize("m,n", [(65, 65), (100, 128), (130, 130), (300, 300), (600, 650), (1500, 140)])
def test_large_multipliers_without_pivoting(handle, dtype, m, n):
    rng = np.random.default_rng(m + n)
    k = min(m, n)
    lo, up = exact_factors(rng, max(m, n), dtype)
    lo, up = lo[:m, :k], up[:k, :n]
    a = lo @ up
    assert np.abs(np.real(a)).max() < 2 ** 23 and np.array_equal(a.astype(dtype), a)
    lu, _ = factor(handle, a.astype(dtype), pivoting=False)
    got_lo, got_up = parts(lu)
    assert np.array_equal(got_up, up)
    assert np.array_equal(got_lo, lo)


@pytest.mark.parametrize("dtype", KINDS)
@pytest.mark.parametrize("n", [100, 128, 600])
def test_rows_above_an_overflow(handle, dtype, n):
    """The product of one multiplier and one entry of U overflows in the last column: the rows of
    that column above it, and all other columns, are exact."""
    a = np.eye(n)
    a[:, n - 1] += np.arange(n) % 5
    a[n - 1, n - 1] = 1
    a[40, 10] = a[10, n - 1] = 2.0 ** 100
    lu, _ = factor(handle, a.astype(dtype), pivoting=False)
    want = a.astype(dtype)
    assert np.array_equal(lu[:, :n - 1], want[:, :n - 1])
    assert np.array_equal(lu[:40, n - 1], want[:40, n - 1])
    assert not np.isfinite(lu[40, n - 1])
