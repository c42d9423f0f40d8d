"""Batched complex inverses of orders 33..64 (one wave per matrix, eight columns a block):
remainders of the blocks, leading dimensions, ties, a singular member."""
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


def invert(torch, a, lda, ldc):
    batch, n, _ = a.shape
    da = np.zeros((batch, n, lda), np.complex64)
    da[:, :, :n] = a.transpose(0, 2, 1)
    ta = torch.from_numpy(da).cuda()
    tc = torch.full((batch, n, ldc), 7, dtype=torch.complex64, device="cuda")
    pa = torch.tensor([ta[i].data_ptr() for i in range(batch)], dtype=torch.int64, device="cuda")
    pc = torch.tensor([tc[i].data_ptr() for i in range(batch)], dtype=torch.int64, device="cuda")
    info = torch.full((batch,), -9, dtype=torch.int32, device="cuda")
    with A.Handle() as h:
        assert A.lib().aclsolverCmatinvBatched(h.h, n, A.ptr(pa), lda, A.ptr(pc), ldc, A.ptr(info), batch) == A.SUCCESS
        torch.cuda.synchronize()
    out = tc.cpu().numpy()
    assert (out[:, :, n:] == 7).all()
    return out[:, :, :n].transpose(0, 2, 1), info.cpu().numpy()


@pytest.mark.parametrize("n", [33, 39, 40, 41, 48, 57, 63, 64])
def test_inverses(torch, n):
    """|X - inv(A)| <= 16 n eps |inv(A)| |A| |inv(A)| in the Frobenius norm (Gauss-Jordan with
    partial pivoting of a random matrix errs by a small multiple of sqrt(n) eps times that)."""
    rng = np.random.default_rng(n)
    a = ((rng.standard_normal((5, n, n)) + 1j * rng.standard_normal((5, n, n))) / np.sqrt(n)).astype(np.complex64)
    a[3] = np.eye(n)[rng.permutation(n)] * (1 + 2j)  # every score of a column but one is zero
    x, info = invert(torch, a, n + 1, n + 2)
    assert (info == 0).all()
    for i in range(5):
        want = np.linalg.inv(a[i].astype(np.complex128))
        size = np.linalg.norm(want)
        assert np.linalg.norm(x[i] - want) <= 16 * n * EPS * size * size * np.linalg.norm(a[i], 2)


@pytest.mark.parametrize("n", [37, 64])
def test_singular_members(torch, n):
    """info is the first zero pivot's step; the other members are not touched by it."""
    rng = np.random.default_rng(n)
    a = (rng.standard_normal((3, n, n)) + 1j * rng.standard_normal((3, n, n))).astype(np.complex64)
    a[0, :, 0] = 0
    a[2, :, 20] = 0
    x, info = invert(torch, a, n, n)
    assert info.tolist() == [1, 0, 21]
    want = np.linalg.inv(a[1].astype(np.complex128))
    assert np.linalg.norm(x[1] - want) <= 16 * n * EPS * np.linalg.norm(want) ** 2 * np.linalg.norm(a[1], 2)


def test_ties_take_the_lowest_row(torch):
    """Entries +-1, +-1j tie in the first column; the row order of the pivots shows only in
    rounding, so the inverse of an exactly representable case is exact."""
    n = 64
    a = np.kron(np.array([[1, 1], [1, -1]]), np.eye(32)).astype(np.complex64) * 1j
    x, info = invert(torch, np.stack([a, a]), n, n)
    assert (info == 0).all()
    assert np.array_equal(x[0], np.linalg.inv(a.astype(np.complex128)).astype(np.complex64)) and np.array_equal(x[0], x[1])
