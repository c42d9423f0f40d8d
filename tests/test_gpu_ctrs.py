"""Chained complex solves (device cgetrs): block edges, strips of right-hand sides, all three
transposes, and a block with a zero pivot."""
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


def factors(n, rng):
    """Packed L, U of moderate condition (both below about 10), and pivots."""
    z = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) / (4 * np.sqrt(n))
    lu = (np.tril(z, -1) + np.triu(z, 1) + np.diag(2 * np.exp(1j * rng.uniform(0, 6, n)))).astype(np.complex64)
    piv = np.array([rng.integers(j, n) + 1 for j in range(n)], np.int32)
    return lu, piv


def solve(torch, lu, piv, b, trans, lda, ldb):
    n, nrhs = b.shape
    da = np.zeros((n, lda), np.complex64)
    da[:, :n] = lu.T
    db = np.full((nrhs, ldb), 7, np.complex64)
    db[:, :n] = b.T
    ta, tb = torch.from_numpy(da).cuda(), torch.from_numpy(db).cuda()
    tp = None if piv is None else torch.from_numpy(piv).cuda()
    info = torch.full((1,), -9, dtype=torch.int32, device="cuda")
    with A.Handle() as h:
        assert A.lib().aclsolverCgetrsDevice(h.h, trans, n, nrhs, A.ptr(ta), lda, None if tp is None else A.ptr(tp),
                                             A.ptr(tb), ldb, A.ptr(info)) == A.SUCCESS
        torch.cuda.synchronize()
    out = tb.cpu().numpy()
    assert (out[:, n:] == 7).all() and int(info[0]) == 0
    return out[:, :n].T


@pytest.mark.parametrize("trans", [0, 1, 2])
@pytest.mark.parametrize("n,nrhs,pivots", [(1, 1, True), (63, 17, True), (64, 16, True), (65, 1, True), (129, 33, False),
                                           (257, 2, True), (700, 5, True), (70, 2048, True), (70, 2049, True)])
def test_solutions(torch, n, nrhs, pivots, trans):
    """Against FP64 on the same factors. Errors of a solve grow like sqrt(n) eps times the
    factors' conditions (below 10 each, most columns far below): 64 sqrt(n + 8) eps."""
    rng = np.random.default_rng(1000 * n + nrhs + trans)
    lu, piv = factors(n, rng)
    x = (rng.standard_normal((n, nrhs)) + 1j * rng.standard_normal((n, nrhs)))
    w = lu.astype(np.complex128)
    pa = (np.tril(w, -1) + np.eye(n)) @ np.triu(w)
    perm = np.arange(n)
    if pivots:
        for j, p in enumerate(piv):
            perm[[j, p - 1]] = perm[[p - 1, j]]
    a = np.empty_like(pa)
    a[perm] = pa
    m = {0: a, 1: a.T, 2: a.conj().T}[trans]
    b = (m @ x).astype(np.complex64)
    want = np.linalg.solve(m, b.astype(np.complex128))
    got = solve(torch, lu, piv if pivots else None, b, trans, n + n % 2, n + 1)
    assert np.linalg.norm(got - want) <= 64 * np.sqrt(n + 8) * EPS * np.linalg.norm(want)


@pytest.mark.parametrize("trans", [0, 2])
def test_zero_pivot(torch, trans):
    """A zero on U's diagonal: the rows that the substitution finishes before it meets the zero
    stay exact to the bound, and the others are not finite."""
    n, at = 150, 100
    rng = np.random.default_rng(trans)
    lu, _ = factors(n, rng)
    lu[at, at] = 0
    w = lu.astype(np.complex128)
    lo, up = np.tril(w, -1) + np.eye(n), np.triu(w)
    b = (rng.standard_normal((n, 1)) + 1j * rng.standard_normal((n, 1))).astype(np.complex64)
    got = solve(torch, lu, None, b, trans, n, n)
    if trans == 0:
        y = np.linalg.solve(lo, b.astype(np.complex128))
        want = np.linalg.solve(up[at + 1:, at + 1:], y[at + 1:])
        assert np.linalg.norm(got[at + 1:] - want) <= 64 * np.sqrt(n + 8) * EPS * np.linalg.norm(want)
        assert not np.isfinite(got[: at + 1]).any()
    else:
        assert not np.isfinite(got[at]).any()
