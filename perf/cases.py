"""Performance cases of the MI355X LU library: the calls that users make, over their real range.

A case is a plain dict with a "kind" and its sizes:

  solve         aclsolverSgetrf + aclsolverSgetrsDevice: factor one real system and solve it
  factor        aclsolverSgetrf of a tall, thin matrix
  gesv          aclsolverSB/SH/SSgesv: the mixed-precision (or FP32) solver with refinement
  inverse       aclsolverSgetrf + aclsolverSgetri
  matinv        aclsolverSmatinvStridedBatched: contiguous batch of small inverses, with pivots
  getri_batched aclsolverSgetriBatched: inverses of a batch from its LU factors
  uneven        aclsolverSgesvVbatched: thousands of systems of different orders through one plan
  csolve        aclsolverCgetrf + aclsolverCgetrsDevice: one complex system
  cmatinv       aclsolverCmatinvBatched: batch of small complex inverses (pointer arrays)

The systems are G / sqrt(n) + s P, with G Gaussian, s = 2 (real) or 1.5 (complex) and P a
random permutation: well conditioned, with the rows in no particular order, so that nearly
every column interchanges rows. Factorizations work in place, so a pass first copies the
matrix, as a program does that still needs it afterwards.
"""
import ctypes
import functools
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "ops-solver_amd"))

import aclsolver  # noqa: E402

REAL_SHIFT, COMPLEX_SHIFT = 2.0, 1.5


def listed():
    return [
        # The smallest dense call: a small coupled system solved inside a larger program, where
        # launches and host round trips are all there is.
        {"name": "solve_64", "kind": "solve", "n": 64, "nrhs": 1, "trans": 0},
        # An ordinary dense system (the benchmark's small dense workload).
        {"name": "solve_512", "kind": "solve", "n": 512, "nrhs": 1, "trans": 0},
        # A larger system of ragged order, several right-hand sides, transposed (adjoint) solve.
        {"name": "solve_2100_t", "kind": "solve", "n": 2100, "nrhs": 16, "trans": 1},
        # A tall and thin factorization: basis selection or one block column of a larger program.
        {"name": "factor_8200x300", "kind": "factor", "m": 8200, "n": 300},
        # The headline: a large dense solve with split-BF16 trailing updates and refinement.
        {"name": "gesv_sb_16384", "kind": "gesv", "mode": "SB", "n": 16384, "nrhs": 1},
        # The same family at a middle, odd-tiled size, FP16 operands.
        {"name": "gesv_sh_4700", "kind": "gesv", "mode": "SH", "n": 4700, "nrhs": 1},
        # An explicit inverse of a ragged matrix from its factors.
        {"name": "inverse_1000", "kind": "inverse", "n": 1000},
        # A large batch of small inverses (the benchmark's batched workload).
        {"name": "matinv_32x65536", "kind": "matinv", "n": 32, "batch": 65536},
        # A batch of middle-sized inverses from existing factors, drop-in pointer arrays.
        {"name": "getri_batched_128x512", "kind": "getri_batched", "n": 128, "batch": 512},
        # Thousands of systems of orders 8..256 (the benchmark's uneven batch).
        {"name": "uneven_20000", "kind": "uneven", "count": 20000, "low": 8, "high": 256, "nrhs": 4},
        # A large complex system with several right-hand sides (the benchmark's complex workload).
        {"name": "csolve_8192", "kind": "csolve", "n": 8192, "nrhs": 16, "trans": 0},
        # A batch of small complex inverses (channel or impedance matrices).
        {"name": "cmatinv_64x4096", "kind": "cmatinv", "n": 64, "batch": 4096},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "factor", "gesv", "inverse", "matinv", "getri_batched", "uneven", "csolve",
                       "cmatinv"])
    if kind == "solve":
        return {"kind": kind, "n": _log_int(rng, 32, 4100), "nrhs": rng.choice([1, 1, 2, 7, 16]),
                "trans": rng.choice([0, 1])}
    if kind == "factor":
        return {"kind": kind, "m": _log_int(rng, 1100, 16384), "n": _log_int(rng, 40, 400)}
    if kind == "gesv":
        return {"kind": kind, "mode": rng.choice(["SB", "SH", "SS"]), "n": _log_int(rng, 500, 9000),
                "nrhs": rng.choice([1, 1, 3])}
    if kind == "inverse":
        return {"kind": kind, "n": _log_int(rng, 100, 2300)}
    if kind == "matinv":
        n = rng.randint(4, 64)
        return {"kind": kind, "n": n, "batch": _log_int(rng, 512, (1 << 26) // (n * n))}
    if kind == "getri_batched":
        n = _log_int(rng, 8, 512)
        return {"kind": kind, "n": n, "batch": _log_int(rng, 4, max(8, (1 << 30) // (n * n * max(n, 64))))}
    if kind == "uneven":
        high = rng.randint(32, 256)
        return {"kind": kind, "count": _log_int(rng, 200, 20000), "low": rng.randint(2, high // 2), "high": high,
                "nrhs": rng.randint(1, 4)}
    if kind == "csolve":
        return {"kind": kind, "n": _log_int(rng, 64, 4100), "nrhs": rng.choice([1, 5, 16]),
                "trans": rng.choice([0, 1, 2])}
    n = rng.randint(4, 64)
    return {"kind": kind, "n": n, "batch": _log_int(rng, 256, (1 << 24) // (n * n))}


# ---------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------


@functools.lru_cache(maxsize=None)
def _handle():
    """The one handle that a program keeps for all its calls."""
    return aclsolver.Handle()


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, cplx, *shape):
    if not cplx:
        return torch.randn(*shape, device="cuda", generator=g)
    return torch.view_as_complex(torch.randn(*shape, 2, device="cuda", generator=g)) * 0.5 ** 0.5


def _matrix(g, m, n, cplx=False):
    """Column-major m x n matrix as a tensor (n, m): element (r, c) is t[c, r]."""
    t = _randn(g, cplx, n, m).mul_(1.0 / math.sqrt(min(m, n)))
    k = min(m, n)
    rows = torch.randperm(m, device="cuda", generator=g)[:k]
    t[torch.arange(k, device="cuda"), rows] += COMPLEX_SHIFT if cplx else REAL_SHIFT
    return t


def _batch(g, batch, n, cplx=False):
    """batch column-major n x n matrices, contiguous: element (r, c) of matrix i is t[i, c, r]."""
    t = _randn(g, cplx, batch, n, n).mul_(1.0 / math.sqrt(n))
    rows = torch.rand(batch, n, device="cuda", generator=g).argsort(dim=1).unsqueeze(2)
    shift = torch.full((batch, n, 1), COMPLEX_SHIFT if cplx else REAL_SHIFT, device="cuda")
    (torch.view_as_real(t)[..., 0] if cplx else t).scatter_add_(2, rows, shift)
    return t


def _sizes(case):
    """The orders of an uneven batch: part of the case, the same for every seed of its inputs."""
    g = torch.Generator()
    g.manual_seed(case["count"] * 1000003 + case["low"] * 1009 + case["high"])
    return torch.randint(case["low"], case["high"] + 1, (case["count"],), generator=g, dtype=torch.int32)


def _uneven(case, seed):
    """Flat matrices and right-hand sides of an uneven batch, with their element offsets."""
    g = _gen(seed)
    n = _sizes(case).cuda().long()
    zero = torch.zeros(1, dtype=torch.long, device="cuda")
    off_a, off_b, off_p = (torch.cat([zero, v.cumsum(0)]) for v in (n * n, n * case["nrhs"], n))
    a = torch.randn(int(off_a[-1]), device="cuda", generator=g)
    a.mul_(torch.repeat_interleave(n.float().rsqrt(), n * n))
    # one shifted row per column, in a random order within each matrix
    ids = torch.repeat_interleave(torch.arange(case["count"], device="cuda"), n)
    keys = ids + torch.rand(ids.numel(), device="cuda", generator=g, dtype=torch.float64)
    row = keys.argsort() - off_p[:-1][ids]
    col = torch.arange(ids.numel(), device="cuda") - off_p[:-1][ids]
    a[off_a[:-1][ids] + col * n[ids] + row] += REAL_SHIFT
    b = torch.randn(int(off_b[-1]), device="cuda", generator=g)
    return n, a, b, off_a, off_b, off_p


class _Plan:
    """An uneven-batch plan, given back with the state that holds it."""

    def __init__(self, case):
        self.sizes = _sizes(case).numpy()
        self.p = ctypes.c_void_p(None)
        _ok(aclsolver.lib().aclsolverSgesvVbatched_createPlan(_handle().h, case["count"], self.sizes.ctypes.data,
                                                              case["nrhs"], ctypes.byref(self.p)))

    def __del__(self):
        if self.p:
            aclsolver.lib().aclsolverSgesvVbatched_destroyPlan(self.p)


def _ok(status):
    if status != aclsolver.SUCCESS:
        raise RuntimeError(f"status {status}")


def _ints(n):
    return torch.empty(n, dtype=torch.int32, device="cuda")


def _pointers(t, stride):
    step = stride * t.element_size()
    return t.data_ptr() + torch.arange(t.shape[0], device="cuda", dtype=torch.int64) * step


def _lwork(fn, *args):
    n = ctypes.c_int(0)
    _ok(fn(_handle().h, *args, ctypes.byref(n)))
    return n.value


def prepare(case, seed):
    L, h, ptr = aclsolver.lib(), _handle().h, aclsolver.ptr
    kind, g = case["kind"], _gen(seed)
    s = {"kind": kind}
    if kind in ("solve", "csolve"):
        cplx, n, nrhs = kind == "csolve", case["n"], case["nrhs"]
        a0, b0 = _matrix(g, n, n, cplx), _randn(g, cplx, nrhs, n)
        a, b, ipiv, info, info2 = torch.empty_like(a0), torch.empty_like(b0), _ints(n), _ints(1), _ints(1)
        getrf = L.aclsolverCgetrf if cplx else L.aclsolverSgetrf
        getrs = L.aclsolverCgetrsDevice if cplx else L.aclsolverSgetrsDevice
        size = L.aclsolverCgetrf_bufferSize if cplx else L.aclsolverSgetrf_bufferSize
        work = torch.empty(max(_lwork(size, n, n, ptr(a), n), 1), dtype=a.dtype, device="cuda")
        s.update(copies=[(a, a0), (b, b0)], keep=work,
                 calls=[(getrf, (h, n, n, ptr(a), n, ptr(work), ptr(ipiv), ptr(info))),
                        (getrs, (h, case["trans"], n, nrhs, ptr(a), n, ptr(ipiv), ptr(b), n, ptr(info2)))],
                 out={"lu": a, "x": b, "ipiv": ipiv, "info_getrf": info, "info_getrs": info2})
    elif kind == "factor":
        m, n = case["m"], case["n"]
        a0 = _matrix(g, m, n)
        a, ipiv, info = torch.empty_like(a0), _ints(min(m, n)), _ints(1)
        work = torch.empty(max(_lwork(L.aclsolverSgetrf_bufferSize, m, n, ptr(a), m), 1), device="cuda")
        s.update(copies=[(a, a0)], keep=work,
                 calls=[(L.aclsolverSgetrf, (h, m, n, ptr(a), m, ptr(work), ptr(ipiv), ptr(info)))],
                 out={"lu": a, "ipiv": ipiv, "info": info})
    elif kind == "gesv":
        n, nrhs = case["n"], case["nrhs"]
        a, b = _matrix(g, n, n), _randn(g, False, nrhs, n)
        x, ipiv, info, size, iters = torch.empty_like(b), _ints(n), _ints(1), ctypes.c_size_t(0), ctypes.c_int(0)
        _ok(getattr(L, f"aclsolver{case['mode']}gesv_bufferSize")(h, n, nrhs, ctypes.byref(size)))
        work = torch.empty(size.value, dtype=torch.uint8, device="cuda")
        s.update(copies=[], keep=(a, b, work), iters=iters,
                 calls=[(getattr(L, f"aclsolver{case['mode']}gesv"),
                         (h, n, nrhs, ptr(a), n, ptr(ipiv), ptr(b), n, ptr(x), n, ptr(work), size.value,
                          ctypes.byref(iters), ptr(info)))],
                 out={"x": x, "ipiv": ipiv, "info": info})
    elif kind == "inverse":
        n = case["n"]
        a0 = _matrix(g, n, n)
        a, ipiv, info, info2 = torch.empty_like(a0), _ints(n), _ints(1), _ints(1)
        work = torch.empty(max(_lwork(L.aclsolverSgetrf_bufferSize, n, n, ptr(a), n), 1), device="cuda")
        lw2 = _lwork(L.aclsolverSgetri_bufferSize, n, ptr(a), n)
        work2 = torch.empty(max(lw2, 1), device="cuda")
        s.update(copies=[(a, a0)], keep=(work, work2),
                 calls=[(L.aclsolverSgetrf, (h, n, n, ptr(a), n, ptr(work), ptr(ipiv), ptr(info))),
                        (L.aclsolverSgetri, (h, n, ptr(a), n, ptr(ipiv), ptr(work2), lw2, ptr(info2)))],
                 out={"inverse": a, "ipiv": ipiv, "info_getrf": info, "info_getri": info2})
    elif kind == "matinv":
        n, batch = case["n"], case["batch"]
        a = _batch(g, batch, n)
        c, ipiv, info = torch.empty_like(a), _ints((batch, n)), _ints(batch)
        s.update(copies=[], keep=a,
                 calls=[(L.aclsolverSmatinvStridedBatched, (h, n, ptr(a), n, n * n, ptr(c), n, n * n, ptr(ipiv),
                                                            ptr(info), batch))],
                 out={"inverse": c, "ipiv": ipiv, "info": info})
    elif kind == "getri_batched":
        n, batch = case["n"], case["batch"]
        lu, piv = torch.linalg.lu_factor(_batch(g, batch, n).transpose(1, 2))
        lu = lu.transpose(1, 2).contiguous()  # column-major factors
        piv, c, info = piv.to(torch.int32).contiguous(), torch.empty_like(lu), _ints(batch)
        pa, pc = _pointers(lu, n * n), _pointers(c, n * n)
        s.update(copies=[], keep=(lu, piv, pa, pc),
                 calls=[(L.aclsolverSgetriBatched, (h, n, ptr(pa), n, ptr(piv), ptr(pc), n, ptr(info), batch))],
                 out={"inverse": c, "info": info})
    elif kind == "uneven":
        n, a0, b0, off_a, off_b, off_p = _uneven(case, seed)
        a, b, ipiv, info = torch.empty_like(a0), torch.empty_like(b0), _ints(int(off_p[-1])), _ints(case["count"])
        pa, pb = a.data_ptr() + 4 * off_a[:-1], b.data_ptr() + 4 * off_b[:-1]
        plan = _Plan(case)
        s.update(copies=[(a, a0), (b, b0)], keep=(pa, pb, plan),
                 calls=[(L.aclsolverSgesvVbatched_execute, (h, plan.p, ptr(pa), ptr(pb), ptr(ipiv), ptr(info)))],
                 out={"lu": a, "x": b, "ipiv": ipiv, "info": info})
    elif kind == "cmatinv":
        n, batch = case["n"], case["batch"]
        a = _batch(g, batch, n, True)
        c, info = torch.empty_like(a), _ints(batch)
        pa, pc = _pointers(a, n * n), _pointers(c, n * n)
        s.update(copies=[], keep=(a, pa, pc),
                 calls=[(L.aclsolverCmatinvBatched, (h, n, ptr(pa), n, ptr(pc), n, ptr(info), batch))],
                 out={"inverse": c, "info": info})
    else:
        raise ValueError(kind)
    return s


def run(state):
    for dst, src in state["copies"]:
        dst.copy_(src)
    for fn, args in state["calls"]:
        _ok(fn(*args))
    if "iters" in state:
        return dict(state["out"], iterations=state["iters"].value)
    return state["out"]


# ---------------------------------------------------------------------------------------
# the least work of a pass, and the outputs in 64 bits
# ---------------------------------------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind in ("solve", "csolve"):
        n, r, c = case["n"], case["nrhs"], 2 if kind == "csolve" else 1
        return {"bytes": c * 8.0 * (n * n + n * r) + 4 * n, "flops": (4 if c == 2 else 1) * (2 / 3 * n ** 3 + 2.0 * n * n * r)}
    if kind == "factor":
        m, n = case["m"], case["n"]
        k = min(m, n)
        return {"bytes": 8.0 * m * n + 4 * k, "flops": 2.0 * m * n * k - (m + n) * float(k) ** 2 + 2 / 3 * float(k) ** 3}
    if kind == "gesv":
        n, r = case["n"], case["nrhs"]
        return {"bytes": 4.0 * n * n + 8.0 * n * r, "flops": 2 / 3 * float(n) ** 3 + 2.0 * n * n * r}
    if kind == "inverse":
        n = case["n"]
        return {"bytes": 8.0 * n * n + 4 * n, "flops": 2.0 * n ** 3}
    if kind == "matinv":
        n, k = case["n"], case["batch"]
        return {"bytes": k * (8.0 * n * n + 4 * n + 4), "flops": k * 2.0 * n ** 3}
    if kind == "getri_batched":
        n, k = case["n"], case["batch"]
        return {"bytes": k * (8.0 * n * n + 4 * n + 4), "flops": k * 4 / 3 * n ** 3}
    if kind == "uneven":
        n, r = _sizes(case).double(), case["nrhs"]
        return {"bytes": float((8 * (n * n + n * r) + 4 * n + 4).sum()),
                "flops": float((2 / 3 * n ** 3 + 2 * n * n * r).sum())}
    n, k = case["n"], case["batch"]
    return {"bytes": k * (16.0 * n * n + 4), "flops": k * 8.0 * n ** 3}


# Factors come from the CPU's LAPACK: it pivots on the largest entry of each column, which the
# GPU's own 64-bit routine does not do at every order.
def _solve64(at, bt, trans):
    """LU and solution in 64 bits of the column-major tensors at (n, n) and bt (nrhs, n)."""
    wide = torch.complex128 if at.is_complex() else torch.float64
    lu, piv = torch.linalg.lu_factor(at.cpu().to(wide).T)
    b = bt.cpu().to(wide).T
    if trans == 1 and at.is_complex():
        x = torch.linalg.lu_solve(lu, piv, b.conj().resolve_conj(), adjoint=True).conj().resolve_conj()
    else:
        x = torch.linalg.lu_solve(lu, piv, b, adjoint=trans != 0)
    return lu.T.contiguous(), x.T.contiguous()


def exact(case, seed):
    kind, g = case["kind"], _gen(seed)
    if kind in ("solve", "csolve"):
        cplx = kind == "csolve"
        a, b = _matrix(g, case["n"], case["n"], cplx), _randn(g, cplx, case["nrhs"], case["n"])
        lu, x = _solve64(a, b, case["trans"])
        return {"lu": lu, "x": x, "ipiv": None, "info_getrf": None, "info_getrs": None}
    if kind == "factor":
        a = _matrix(g, case["m"], case["n"]).cpu().double()
        lu, _ = torch.linalg.lu_factor(a.T)
        return {"lu": lu.T.contiguous(), "ipiv": None, "info": None}
    if kind == "gesv":
        a, b = _matrix(g, case["n"], case["n"]), _randn(g, False, case["nrhs"], case["n"])
        return {"x": torch.linalg.solve(a.double().T, b.double().T).T.contiguous(), "ipiv": None, "info": None, "iterations": None}
    if kind == "inverse":
        a = _matrix(g, case["n"], case["n"]).double()
        return {"inverse": torch.linalg.inv(a), "ipiv": None, "info_getrf": None, "info_getri": None}
    if kind == "matinv":
        return {"inverse": torch.linalg.inv(_batch(g, case["batch"], case["n"]).double()), "ipiv": None, "info": None}
    if kind == "getri_batched":
        n = case["n"]
        lu, piv = torch.linalg.lu_factor(_batch(g, case["batch"], n).transpose(1, 2))
        eye = torch.eye(n, dtype=torch.float64, device="cuda").expand_as(lu)
        inv = torch.linalg.lu_solve(lu.double(), piv, eye)
        return {"inverse": inv.transpose(1, 2).contiguous(), "info": None}
    if kind == "uneven":
        n, a, b, off_a, off_b, _ = (v.cpu() for v in _uneven(case, seed))
        lu, x, r = torch.empty_like(a, dtype=torch.float64), torch.empty_like(b, dtype=torch.float64), case["nrhs"]
        for k in n.unique().tolist():  # all systems of one order at a time
            which = (n == k).nonzero().flatten()
            ia = off_a[which][:, None] + torch.arange(k * k)
            ib = off_b[which][:, None] + torch.arange(k * r)
            f, p = torch.linalg.lu_factor(a[ia].double().view(-1, k, k).transpose(1, 2))
            lu[ia] = f.transpose(1, 2).reshape(len(which), -1)
            y = torch.linalg.lu_solve(f, p, b[ib].double().view(-1, r, k).transpose(1, 2))
            x[ib] = y.transpose(1, 2).reshape(len(which), -1)
        return {"lu": lu, "x": x, "ipiv": None, "info": None}
    a = _batch(g, case["batch"], case["n"], True).to(torch.complex128)
    return {"inverse": torch.linalg.inv(a), "info": None}
