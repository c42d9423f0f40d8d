"""Uneven batched solves, orders 65..256: the one-workgroup-per-matrix kernels against the
column-cyclic ones (which a plan with its own schedule takes), at the edges of the wave classes,
panels, blocks of eight columns and right-hand sides; singular, tied and NaN members."""
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
SIZES = [65, 66, 71, 72, 73, 124, 125, 127, 128, 129, 130, 136, 188, 191, 192, 193, 200, 249, 252, 253, 255, 256]


def _run(torch, mats, rhs, nrhs, schedule):
    """Each system as many times as fills its class (one-workgroup kernels are for full devices); the
    copies have to agree bit for bit, the first of each comes back."""
    copies = [1 if schedule is not None else 146 if m.shape[0] > 192 else 210 if m.shape[0] > 128 else 227 for m in mats]
    start = np.concatenate([[0], np.cumsum(copies)])
    sizes = np.repeat(np.array([m.shape[0] for m in mats], np.int32), copies)
    dA, dB = [], []
    for m, b, k in zip(mats, rhs, copies):
        dA += list(torch.from_numpy(np.ascontiguousarray(m.T)).cuda().repeat(k, 1, 1))
        dB += list(torch.from_numpy(np.ascontiguousarray(b.T)).cuda().repeat(k, 1, 1))
    mats = sizes
    pa = torch.tensor([t.data_ptr() for t in dA], dtype=torch.int64, device="cuda")
    pb = torch.tensor([t.data_ptr() for t in dB], dtype=torch.int64, device="cuda")
    ipiv = torch.zeros(int(sizes.sum()), dtype=torch.int32, device="cuda")
    info = torch.full((len(mats),), -9, dtype=torch.int32, device="cuda")
    plan = ctypes.c_void_p(None)
    L = A.lib()
    with A.Handle() as h:
        if schedule is None:
            st = L.aclsolverSgesvVbatched_createPlan(h.h, len(mats), sizes.ctypes.data, nrhs, ctypes.byref(plan))
        else:
            st = L.aclsolverSgesvVbatched_createPlanWithSchedule(h.h, len(mats), sizes.ctypes.data, nrhs,
                                                                 schedule.ctypes.data, ctypes.byref(plan))
        assert st == A.SUCCESS
        assert L.aclsolverSgesvVbatched_execute(h.h, plan, A.ptr(pa), A.ptr(pb), A.ptr(ipiv), A.ptr(info)) == A.SUCCESS
        torch.cuda.synchronize()
        L.aclsolverSgesvVbatched_destroyPlan(plan)
    off = np.concatenate([[0], np.cumsum(sizes)])
    for i, k in enumerate(copies):
        a = torch.stack(dA[start[i]:start[i + 1]]).view(torch.int32)
        assert (a == a[:1]).all() and (info[start[i]:start[i + 1]] == info[start[i]]).all()
    first = start[:-1]
    piv = np.concatenate([ipiv[off[i]:off[i + 1]].cpu().numpy() for i in first])
    return [dA[i].cpu().numpy().T for i in first], [dB[i].cpu().numpy().T for i in first], piv, info.cpu().numpy()[first]


@pytest.mark.parametrize("nrhs", [0, 1, 2, 3, 4])
def test_against_the_column_cyclic_kernels(nrhs):
    """Pivots and info equal; factors and solutions differ by rounding only: both paths subtract
    the same products, 8 n eps of the largest factor entry (times the growth of the solve, at most
    64 for these shifted matrices) bounds any difference in their order."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(70 + nrhs)
    mats, rhs = [], []
    for i, n in enumerate(SIZES):
        a = (rng.standard_normal((n, n)) / np.sqrt(n)).astype(np.float32)
        a[rng.permutation(n), np.arange(n)] += 2
        if i % 5 == 1:  # ties: the lowest row wins
            a[:, 0] = np.where(rng.random(n) < 0.5, 1, -1)
        if i % 5 == 2:  # a zero column in the second panel
            a[:, 64] = 0
        if i % 5 == 3:  # a NaN off the diagonal loses, its row is spoiled
            a[n - 1, 3] = np.nan
        mats.append(a)
        rhs.append(rng.standard_normal((n, max(nrhs, 1))).astype(np.float32))
    schedule = np.array([1] * 4 + [3] * 4 + [5] * 4, np.int32)
    lu, x, piv, info = _run(torch, mats, rhs, nrhs, None)
    lu0, x0, piv0, info0 = _run(torch, mats, rhs, nrhs, schedule)
    assert np.array_equal(info, info0)
    at = 0
    for i, n in enumerate(SIZES):
        if i % 5 != 3:  # beyond a NaN row the pivots of both paths are arbitrary
            assert np.array_equal(piv[at:at + n], piv0[at:at + n]), n
            assert info[i] == (65 if i % 5 == 2 and n > 64 else 0)
        at += n
        if i % 5 in (0, 1, 4):
            assert np.abs(lu[i] - lu0[i]).max() <= 8 * n * EPS * np.abs(lu0[i]).max()
            assert np.abs(x[i] - x0[i]).max() <= 64 * 8 * n * EPS * np.abs(x0[i]).max()
        elif i % 5 == 2:  # U above the zero column is defined
            assert np.abs(lu[i][:, :64] - lu0[i][:, :64]).max() <= 8 * n * EPS * np.abs(lu0[i][:, :64]).max()
