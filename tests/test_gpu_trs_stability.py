"""Device solves from factors whose triangular blocks have large inverses: results as from a
substitution."""
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
# A type and the forms of op(A) that it has.
FORMS = [(np.float32, 0), (np.float32, 1), (np.complex64, 0), (np.complex64, 1), (np.complex64, 2)]


@pytest.fixture(scope="module")
def handle():
    h = A.Handle()
    yield h
    h.close()


def operators(lo, up, trans):
    """The two triangles of op(A) in the order of their solves."""
    if trans == 0:
        return lo, up
    f = np.conj if trans == 2 else (lambda x: x)
    return f(up).T, f(lo).T


def solve(handle, packed, b, trans):
    import torch

    n, nrhs = b.shape
    print(f"getrs {packed.dtype} n={n} nrhs={nrhs} trans={trans}", flush=True)
    ipiv = torch.arange(1, n + 1, dtype=torch.int32, device="cuda")
    d, x = A.to_device_cm(packed), A.to_device_cm(b)
    info = torch.full((1,), 7, dtype=torch.int32, device="cuda")
    getrs = A.lib().aclsolverCgetrsDevice if packed.dtype == np.complex64 else A.lib().aclsolverSgetrsDevice
    assert getrs(handle.h, trans, n, nrhs, A.ptr(d), n, A.ptr(ipiv), A.ptr(x), n, A.ptr(info)) == A.SUCCESS
    torch.cuda.synchronize()
    assert info.item() == 0
    return A.from_device_cm(x, n, nrhs)


@pytest.mark.parametrize("dtype,trans", FORMS)
@pytest.mark.parametrize("nrhs", [1, 5, 40])
@pytest.mark.parametrize("lower", [False, True])
@pytest.mark.parametrize("n", [64, 100, 300])
def test_exact_solutions(handle, dtype, trans, nrhs, lower, n):
    """-1 below L's diagonal, or above U's, and the other factor diagonal (powers of two): with small
    integer solutions every number that a substitution meets is an integer below 2^24, so it is
    exact, while the inverse reaches 2^62 in a block."""
    rng = np.random.default_rng(n + nrhs + trans)
    ones = np.tri(n, k=-1)
    lo = np.eye(n) - (ones if lower else 0)
    up = np.diag(rng.choice([1.0, 2.0], n)) if lower else np.eye(n) - ones.T
    unit = 1j if dtype == np.complex64 else 1
    lo, up = np.eye(n) + (lo - np.eye(n)) * unit, np.diag(np.diag(up)) + np.triu(up, 1) * unit
    t1, t2 = operators(lo, up, trans)
    x0 = rng.integers(-3, 4, (n, nrhs)) * (1 + unit if dtype == np.complex64 else 1)
    b = t1 @ (t2 @ x0)
    packed = (np.tril(lo, -1) + np.triu(up)).astype(dtype)
    assert np.abs(b).max() < 2 ** 22 and np.array_equal(b.astype(dtype), b)
    assert np.array_equal(solve(handle, packed, b.astype(dtype), trans), x0.astype(dtype))
