"""aclsolverSgetri works in the caller's workspace alone: two calls on one handle, with a stream
and a workspace each, do not meet, and every accepted workspace size gives the inverse."""
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


def _system(n, seed):
    rng = np.random.default_rng(seed)
    a = (rng.standard_normal((n, n)) / np.sqrt(n) + 2 * np.eye(n)[rng.permutation(n)]).astype(np.float32)
    lu, piv, info = O.sgetrf(a)
    assert info == 0
    return a, lu, piv


@pytest.mark.parametrize("n", [1, 63, 65, 150, 300])
def test_smallest_and_reported_workspace(n):
    import torch

    a, lu, piv = _system(n, n)
    L = A.lib()
    with A.Handle() as h:
        lw = ctypes.c_int(0)
        info = torch.zeros(1, dtype=torch.int32, device="cuda")
        dpiv = torch.from_numpy(piv).cuda()
        tail = 1024
        assert L.aclsolverSgetri_bufferSize(h.h, n, None, n, ctypes.byref(lw)) == A.SUCCESS
        work = torch.empty(lw.value + tail, device="cuda")

        def call(size):
            d = A.to_device_cm(lu)
            work[size:] = 5.0
            st = L.aclsolverSgetri(h.h, n, A.ptr(d), n, A.ptr(dpiv), A.ptr(work), size, A.ptr(info))
            torch.cuda.synchronize()
            assert bool((work[size:] == 5.0).all())
            return st, d

        lo, hi = 0, lw.value  # refused, accepted
        while hi - lo > 1:
            mid = (lo + hi) // 2
            st, _ = call(mid)
            lo, hi = (lo, mid) if st == A.SUCCESS else (mid, hi)
        assert info.item() in (0, -6)
        for size in (hi, lw.value - 1, lw.value):
            st, d = call(max(size, hi))
            assert st == A.SUCCESS and info.item() == 0
            assert O.inverse_residual(a, A.from_device_cm(d, n, n)) <= 5


def test_two_streams_on_one_handle():
    import torch

    n = 700
    L = A.lib()
    sys_ = [_system(n, s) for s in (1, 2)]
    streams = [torch.cuda.Stream() for _ in range(2)]
    with A.Handle() as h:
        lw = ctypes.c_int(0)
        assert L.aclsolverSgetri_bufferSize(h.h, n, None, n, ctypes.byref(lw)) == A.SUCCESS
        work = [torch.empty(lw.value, device="cuda") for _ in range(2)]
        info = torch.full((2,), 7, dtype=torch.int32, device="cuda")

        def run(order):
            ds = [A.to_device_cm(lu) for _, lu, _ in sys_]
            torch.cuda.synchronize()
            for k in order:
                L.aclsolverSetStream(h.h, ctypes.c_void_p(streams[k].cuda_stream))
                st = L.aclsolverSgetri(h.h, n, A.ptr(ds[k]), n, None, A.ptr(work[k]), lw.value, info[k:].data_ptr())
                assert st == A.SUCCESS
            torch.cuda.synchronize()
            return ds

        want = [run([k])[k] for k in (0, 1)]
        for _ in range(5):
            got = run([0, 1])
            assert info.tolist() == [0, 0]
            assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
