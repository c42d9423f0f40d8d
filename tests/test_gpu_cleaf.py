"""Complex LU at the edges of its panel kernels: leaves of 64 columns (one workgroup up to 512
rows, then several), the launch that swaps and inverts, the update, the U12 solve and the outer
panels of 512 columns."""
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


@pytest.fixture(scope="module")
def torch():
    t = pytest.importorskip("torch")
    if not t.cuda.is_available():
        pytest.skip("needs a GPU")
    return t


def factor(torch, a, lda=None, pivoting=True):
    m, n = a.shape
    lda = lda or m
    buf = np.zeros((n, lda), np.complex64)
    buf[:, :m] = a.T
    d = torch.from_numpy(buf).cuda()
    piv = torch.zeros(min(m, n), dtype=torch.int32, device="cuda")
    info = torch.full((1,), -9, dtype=torch.int32, device="cuda")
    with A.Handle() as h:
        lw = ctypes.c_int(0)
        assert A.lib().aclsolverCgetrf_bufferSize(h.h, m, n, A.ptr(d), lda, ctypes.byref(lw)) == A.SUCCESS
        work = torch.zeros(lw.value, dtype=torch.complex64, device="cuda")
        assert A.lib().aclsolverCgetrf(h.h, m, n, A.ptr(d), lda, A.ptr(work), A.ptr(piv) if pivoting else None,
                                       A.ptr(info)) == A.SUCCESS
        torch.cuda.synchronize()
    out = d.cpu().numpy()
    assert (out[:, m:] == 0).all()
    return out[:, :m].T, piv.cpu().numpy(), int(info[0])


def l1(x):
    return np.abs(x.real) + np.abs(x.imag)


@pytest.mark.parametrize("m,n", [(1, 1), (2, 3), (63, 63), (64, 64), (65, 65), (128, 128), (129, 130), (256, 256),
                                 (257, 190), (512, 512), (513, 513), (577, 577), (640, 64), (130, 700), (1030, 1030),
                                 (8192, 65), (8193, 66), (16384, 64)])
def test_factors(torch, m, n):
    """|PA - LU| against the a-priori bound 4 (k + 8) eps |L||U| (four real roundings a complex
    product term), in the Frobenius norm; every pivot has its column's largest |re| + |im|."""
    rng = np.random.default_rng(m * 7 + n)
    a = (rng.standard_normal((m, n)) + 1j * rng.standard_normal((m, n))).astype(np.complex64)
    lu, piv, info = factor(torch, a, lda=m + (m % 3))
    k = min(m, n)
    assert info == 0
    perm = np.arange(m)
    for j, p in enumerate(piv):
        assert j + 1 <= p <= m
        perm[[j, p - 1]] = perm[[p - 1, j]]
    lo = np.tril(lu[:, :k].astype(np.complex128), -1) + np.eye(m, k)
    up = np.triu(lu[:k].astype(np.complex128))
    gap = np.linalg.norm(a[perm] - lo @ up)
    assert gap <= 4 * (k + 8) * EPS * np.linalg.norm(np.abs(lo) @ np.abs(up))
    for j in range(k):
        if j + 1 < m:
            assert l1(lo[j + 1:, j] * up[j, j]).max() <= l1(up[j, j]) * (1 + 64 * (k + 8) * EPS) + 64 * (k + 8) * EPS


@pytest.mark.parametrize("m", [60, 100, 500, 700, 9000])
def test_pivot_rule(torch, m):
    """Lowest row on ties, a NaN row last, an overflowing sum still ranked, the first zero column
    in info."""
    rng = np.random.default_rng(m)
    base = (rng.standard_normal((m, 3)) + 1j * rng.standard_normal((m, 3))).astype(np.complex64)
    a = base.copy()
    a[:, 0] = np.where(np.arange(m) % 2 == 0, 1.0, -1.0j)
    assert factor(torch, a)[1][0] == 1
    a = base.copy()
    a[:, 0] = np.nan
    a[m - 2, 0] = 1e-3
    assert factor(torch, a)[1][0] == m - 1
    a = base.copy()
    a[:, 0] = 3e38
    a[m // 2, 0] = 3e38 + 3e38j
    assert factor(torch, a)[1][0] == m // 2 + 1
    a = base.copy()
    a[:, 1] = 2 * a[:, 0]
    a[:, 0] = 0
    lu, piv, info = factor(torch, a)
    assert info == 1 and piv[0] == 1


@pytest.mark.parametrize("n", [65, 600])
def test_without_pivoting(torch, n):
    """No interchanges: the factors of a diagonally dominant matrix, to the same bound."""
    rng = np.random.default_rng(n)
    a = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n)) + 4 * n * np.eye(n)).astype(np.complex64)
    lu, _, info = factor(torch, a, pivoting=False)
    lo = np.tril(lu.astype(np.complex128), -1) + np.eye(n)
    up = np.triu(lu.astype(np.complex128))
    assert info == 0
    assert np.linalg.norm(a - lo @ up) <= 4 * (n + 8) * EPS * np.linalg.norm(np.abs(lo) @ np.abs(up))
