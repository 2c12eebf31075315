"""Timed cases of the dense factor-and-solve path, through the C ABI of libzmlhip.so.

Each case is one call (or the factor-and-solve pair of calls) that a program
using this library makes again and again: matrix products, triangular solves,
LU and Cholesky solves in FP64, the mixed-precision solvers with FP64
refinement, and batches of small systems. Inputs are synthetic and made on the
device from a seed; factorizations overwrite their matrix, so those passes
begin with the copy that a program which still needs A (for its residual, or
for the next time step) makes.
"""
from __future__ import annotations

import ctypes
import math
import random

import numpy as np
import torch

from zml_amd import _lib
from zml_amd._lib import IROpts, IRResult

ROW, COL = 101, 102
TRANS = {"N": 111, "T": 112}
UPLO = {"U": 121, "L": 122}
DIAG = {"N": 131, "U": 132}
SIDE = {"L": 141, "R": 142}
LAYOUT = {"row": ROW, "col": COL}
PRECISION = {"fp32": 0, "fp16": 1, "bf16": 2}


# ---- the cases ----------------------------------------------------------------------
def listed():
    return [
        # the residual product of a refinement written by the caller: one matrix-vector product
        {"name": "gemv_2000", "kind": "gemv", "layout": "row", "trans": "N", "m": 2000, "n": 2000, "beta": 0.0},
        # a product of ordinary, ragged size, one operand transposed (normal equations, projections)
        {"name": "dgemm_ragged", "kind": "gemm", "dtype": "f64", "layout": "row", "ta": "T", "tb": "N",
         "m": 1001, "n": 1500, "k": 777, "beta": 0.0},
        # the FP32 entry at the size of a model layer or an FP32 working copy
        {"name": "sgemm_4096", "kind": "gemm", "dtype": "f32", "layout": "row", "ta": "N", "tb": "N",
         "m": 4096, "n": 4096, "k": 4096, "beta": 0.0},
        # a block of right-hand sides against an existing factor
        {"name": "trsm_4096x1024", "kind": "trsm", "layout": "col", "side": "L", "uplo": "L", "trans": "N",
         "diag": "N", "m": 4096, "n": 1024},
        # the drop-in LAPACKE call on host memory, as an existing program makes it
        {"name": "gesv_host_200", "kind": "gesv_host", "layout": "row", "n": 200, "nrhs": 1},
        # the reference's own small LU configuration, with several right-hand sides
        {"name": "lu_1024", "kind": "lu", "layout": "col", "n": 1024, "nrhs": 16},
        # the plain FP64 LU configuration
        {"name": "lu_16384", "kind": "lu", "layout": "row", "n": 16384, "nrhs": 1},
        # a Cholesky solve of ordinary, ragged size (least squares, Gaussian processes)
        {"name": "chol_1500", "kind": "chol", "layout": "row", "uplo": "U", "n": 1500, "nrhs": 5},
        # the plain FP64 Cholesky configuration
        {"name": "chol_16384", "kind": "chol", "layout": "col", "uplo": "L", "n": 16384, "nrhs": 1},
        # the headline: mixed-precision LU with FP64 refinement of a badly scaled system
        {"name": "mixed_lu_32768", "kind": "mixed_lu", "layout": "row", "n": 32768, "nrhs": 1,
         "precision": "fp16", "delta": 0.1, "decades": 3.0},
        # the mixed-precision Cholesky configuration: 16 right-hand sides
        {"name": "mixed_chol_32768", "kind": "mixed_chol", "layout": "col", "uplo": "L", "n": 32768, "nrhs": 16,
         "precision": "fp16", "mu": 1.0},
        # the batched configuration: 20,000 uneven small systems in one graph launch
        {"name": "batch_20000", "kind": "batch", "count": 20000, "nmin": 8, "nmax": 256},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemm", "trsm", "gesv_host", "lu", "chol", "mixed_lu", "mixed_chol", "batch"])
    layout = rng.choice(["row", "col"])
    if kind == "gemv":
        return {"kind": kind, "layout": layout, "trans": rng.choice("NT"), "m": _log_int(rng, 200, 12000),
                "n": _log_int(rng, 200, 12000), "beta": rng.choice([0.0, 0.5])}
    if kind == "gemm":
        return {"kind": kind, "dtype": rng.choice(["f64", "f64", "f32"]), "layout": layout, "ta": rng.choice("NT"),
                "tb": rng.choice("NT"), "m": _log_int(rng, 64, 6000), "n": _log_int(rng, 64, 6000),
                "k": _log_int(rng, 64, 6000), "beta": rng.choice([0.0, 0.5])}
    if kind == "trsm":
        side = rng.choice("LR")
        tri, other = _log_int(rng, 64, 6000), _log_int(rng, 1, 4000)
        return {"kind": kind, "layout": layout, "side": side, "uplo": rng.choice("UL"), "trans": rng.choice("NT"),
                "diag": rng.choice("NNU"), "m": tri if side == "L" else other, "n": other if side == "L" else tri}
    if kind == "gesv_host":
        return {"kind": kind, "layout": layout, "n": _log_int(rng, 16, 1500), "nrhs": _log_int(rng, 1, 16)}
    if kind == "lu":
        return {"kind": kind, "layout": layout, "n": _log_int(rng, 100, 12000), "nrhs": _log_int(rng, 1, 64)}
    if kind == "chol":
        return {"kind": kind, "layout": layout, "uplo": rng.choice("UL"), "n": _log_int(rng, 100, 12000),
                "nrhs": _log_int(rng, 1, 64)}
    if kind == "mixed_lu":
        return {"kind": kind, "layout": layout, "n": _log_int(rng, 500, 16000), "nrhs": _log_int(rng, 1, 4),
                "precision": rng.choice(["fp16", "fp16", "bf16", "fp32"]), "delta": rng.choice([1.0, 0.1]),
                "decades": rng.choice([0.0, 3.0])}
    if kind == "mixed_chol":
        return {"kind": kind, "layout": layout, "uplo": rng.choice("UL"), "n": _log_int(rng, 500, 16000),
                "nrhs": _log_int(rng, 1, 20), "precision": rng.choice(["fp16", "fp16", "bf16", "fp32"]),
                "mu": rng.choice([1.0, 0.25])}
    return {"kind": "batch", "count": _log_int(rng, 100, 15000), "nmin": 8, "nmax": rng.choice([64, 160, 256])}


# ---- inputs -------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _uniform(g, *shape, dtype=torch.float64):
    return torch.rand(*shape, dtype=dtype, device="cuda", generator=g).mul_(2).sub_(1)


def _stored(M, layout):
    """The logical matrix M as memory in `layout` (a row-major tensor over it) and its leading dimension."""
    T = M.contiguous() if layout == "row" else M.t().contiguous()
    return T, max(1, T.shape[1])


def _logical(T, layout):
    return T if layout == "row" else T.t()


def _general(g, n):
    """A general matrix whose pivots come from anywhere: U[-1, 1] + sqrt(n) I with its rows in random order."""
    A = _uniform(g, n, n)
    A.diagonal().add_(math.sqrt(n))
    return A[torch.randperm(n, generator=g, device="cuda")]


def _spd(g, n, mu, inner):
    B = torch.randn(n, inner, dtype=torch.float64, device="cuda", generator=g)
    A = (B @ B.t()).div_(inner)
    A.diagonal().add_(mu)
    return A.tril_().add_(A.tril(-1).t())


def _scaled(g, n, delta, decades):
    """diag(r) (R + delta n I) diag(c), R ~ U[-0.5, 0.5], r, c = 10^U(-decades, decades)."""
    A = torch.rand(n, n, dtype=torch.float64, device="cuda", generator=g).sub_(0.5)
    A.diagonal().add_(delta * n)
    for dim in (1, 0):
        A.mul_(torch.pow(10.0, _uniform(g, n).mul_(decades)).unsqueeze(dim))
    return A


def _inputs(case, seed):
    """The logical operands of a case, on the device."""
    g, kind = _gen(seed), case["kind"]
    if kind == "gemv":
        A = _uniform(g, case["m"], case["n"])
        nx, ny = (case["n"], case["m"]) if case["trans"] == "N" else (case["m"], case["n"])
        return A, _uniform(g, nx), _uniform(g, ny)
    if kind == "gemm":
        dt = torch.float64 if case["dtype"] == "f64" else torch.float32
        m, n, k = case["m"], case["n"], case["k"]
        A = _uniform(g, *((m, k) if case["ta"] == "N" else (k, m)), dtype=dt)
        B = _uniform(g, *((k, n) if case["tb"] == "N" else (n, k)), dtype=dt)
        return A, B, _uniform(g, m, n, dtype=dt)
    if kind == "trsm":
        q = case["m"] if case["side"] == "L" else case["n"]
        A = _uniform(g, q, q).div_(math.sqrt(q))
        A.diagonal().copy_(torch.rand(q, dtype=torch.float64, device="cuda", generator=g).add_(1))
        return A, _uniform(g, case["m"], case["n"])
    if kind in ("lu", "gesv_host"):
        return _general(g, case["n"]), _uniform(g, case["n"], case["nrhs"])
    if kind == "chol":
        return _spd(g, case["n"], 1.0, case["n"]), _uniform(g, case["n"], case["nrhs"])
    n = case["n"]
    A = _scaled(g, n, case["delta"], case["decades"]) if kind == "mixed_lu" else _spd(g, n, case["mu"], max(1, n // 4))
    x = _uniform(g, n, case["nrhs"])
    return A, A @ x, x


def _batch_sizes(case):
    """Orders, right-hand sides and kinds of a batch (the same for every seed), in groups of equal shape."""
    r = random.Random(case["count"])
    groups = {}
    for i in range(case["count"]):
        key = (_log_int(r, case["nmin"], case["nmax"]), r.randint(1, 4), r.randrange(2))
        groups.setdefault(key, []).append(i)
    return sorted(groups.items())


def _batch_inputs(case, seed):
    """[(n, nrhs, spd, systems, A, B)]: A (count, n, n) and B (count, nrhs, n), column-major systems."""
    g, out = _gen(seed), []
    for (n, nrhs, spd), ids in _batch_sizes(case):
        A = _uniform(g, len(ids), n, n)
        if spd:
            A = torch.bmm(A, A.transpose(1, 2).contiguous()).div_(n)
            A.diagonal(dim1=1, dim2=2).add_(1.0)
        else:
            A.diagonal(dim1=1, dim2=2).add_(n / 4.0)
        out.append((n, nrhs, spd, ids, A, _uniform(g, len(ids), nrhs, n)))
    return out


# ---- prepare ------------------------------------------------------------------------
def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _np(a):
    return a.ctypes.data_as(ctypes.c_void_p)


class _State:
    """What a program holds: the device arrays, the handle of the library and the stream."""

    def __init__(self, case):
        self.case, self.zh = case, _lib.load()
        self.stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        self.plan = None

    def check(self, rc):
        if rc != 0:
            raise RuntimeError("%s: %d %s" % (self.case["kind"], rc, _lib.last_error()))

    def __del__(self):
        if self.plan is not None:
            self.zh.zmlhip_batch_plan_destroy(self.plan)


def _prepare_batch(s, case, seed):
    data = _batch_inputs(case, seed)
    count = case["count"]
    n, nrhs, spd = (np.zeros(count, np.int32) for _ in range(3))
    a, b, x = (np.zeros(count, np.uint64) for _ in range(3))
    s.x = torch.zeros(sum(B.numel() for *_, B in data), dtype=torch.float64, device="cuda")
    s.keep, at = [], 0
    for order, q, kind, ids, A, B in data:
        ids = np.asarray(ids)
        k = np.arange(len(ids), dtype=np.uint64)
        n[ids], nrhs[ids], spd[ids] = order, q, kind
        a[ids] = A.data_ptr() + k * np.uint64(8 * order * order)
        b[ids] = B.data_ptr() + k * np.uint64(8 * order * q)
        x[ids] = s.x.data_ptr() + 8 * at + k * np.uint64(8 * order * q)
        at += B.numel()
        s.keep.append((A, B))
    plan = ctypes.c_void_p()
    torch.cuda.synchronize()
    s.check(s.zh.zmlhip_batch_plan_create(ctypes.byref(plan), count, _np(n), _np(nrhs), _np(spd), _np(a), _np(b),
                                          _np(x), None, 1, s.stream))
    s.plan = plan
    return s


def prepare(case, seed):
    s, kind = _State(case), case["kind"]
    if kind == "batch":
        return _prepare_batch(s, case, seed)
    layout = LAYOUT[case["layout"]]
    ops = _inputs(case, seed)
    if kind == "gemv":
        s.a, lda = _stored(ops[0], case["layout"])
        s.x, s.y = ops[1], ops[2]
        s.args = (layout, TRANS[case["trans"]], case["m"], case["n"], 1.0, _p(s.a), lda, _p(s.x), 1, case["beta"],
                  _p(s.y), 1, s.stream)
    elif kind == "gemm":
        s.a, lda = _stored(ops[0], case["layout"])
        s.b, ldb = _stored(ops[1], case["layout"])
        s.c, ldc = _stored(ops[2], case["layout"])
        s.call = s.zh.zmlhip_dgemm if case["dtype"] == "f64" else s.zh.zmlhip_sgemm
        s.args = (layout, TRANS[case["ta"]], TRANS[case["tb"]], case["m"], case["n"], case["k"], 1.0, _p(s.a), lda,
                  _p(s.b), ldb, case["beta"], _p(s.c), ldc, s.stream)
    elif kind == "trsm":
        s.a, lda = _stored(ops[0], case["layout"])
        s.b0, ldb = _stored(ops[1], case["layout"])
        s.b = torch.empty_like(s.b0)
        s.args = (layout, SIDE[case["side"]], UPLO[case["uplo"]], TRANS[case["trans"]], DIAG[case["diag"]], case["m"],
                  case["n"], 1.0, _p(s.a), lda, _p(s.b), ldb, s.stream)
    elif kind == "gesv_host":
        n, nrhs = case["n"], case["nrhs"]
        (ta, lda), (tb, ldb) = _stored(ops[0], case["layout"]), _stored(ops[1], case["layout"])
        s.a0, s.b0 = ta.cpu().numpy(), tb.cpu().numpy()
        s.a, s.b, s.ipiv = np.empty_like(s.a0), np.empty_like(s.b0), np.zeros(n, np.int32)
        s.args = (layout, n, nrhs, _np(s.a), lda, _np(s.ipiv), _np(s.b), ldb)
    elif kind in ("lu", "chol"):
        n, nrhs = case["n"], case["nrhs"]
        (s.a0, lda), (s.b0, ldb) = _stored(ops[0], case["layout"]), _stored(ops[1], case["layout"])
        s.a, s.b = torch.empty_like(s.a0), torch.empty_like(s.b0)
        s.info = torch.zeros(1, dtype=torch.int32, device="cuda")
        if kind == "lu":
            s.ipiv = torch.zeros(n, dtype=torch.int32, device="cuda")
            s.factor = (layout, n, n, _p(s.a), lda, _p(s.ipiv), _p(s.info), s.stream)
            s.solve = (layout, b"N", n, nrhs, _p(s.a), lda, _p(s.ipiv), _p(s.b), ldb, s.stream)
        else:
            ul = case["uplo"].encode()
            s.factor = (layout, ul, n, _p(s.a), lda, _p(s.info), s.stream)
            s.solve = (layout, ul, n, nrhs, _p(s.a), lda, _p(s.b), ldb, s.stream)
    else:
        n, nrhs = case["n"], case["nrhs"]
        s.a, lda = _stored(ops[0], case["layout"])
        s.b, ldb = _stored(ops[1], case["layout"])
        s.x = torch.zeros_like(s.b)
        s.opts, s.result = IROpts(precision=PRECISION[case["precision"]]), IRResult()
        ul = () if kind == "mixed_lu" else (case["uplo"].encode(),)
        s.call = s.zh.zmlhip_dgesv_mixed if kind == "mixed_lu" else s.zh.zmlhip_dposv_mixed
        s.args = (layout, *ul, n, nrhs, _p(s.a), lda, _p(s.b), ldb, _p(s.x), ldb, ctypes.byref(s.opts),
                  ctypes.byref(s.result), s.stream)
    return s


# ---- one pass -----------------------------------------------------------------------
def run(s):
    kind = s.case["kind"]
    if kind == "gemv":
        s.check(s.zh.zmlhip_dgemv(*s.args))
        return s.y
    if kind == "gemm":
        s.check(s.call(*s.args))
        return s.c
    if kind == "trsm":
        s.b.copy_(s.b0)
        s.check(s.zh.zmlhip_dtrsm(*s.args))
        return s.b
    if kind == "gesv_host":
        np.copyto(s.a, s.a0)
        np.copyto(s.b, s.b0)
        s.check(s.zh.LAPACKE_dgesv(*s.args))
        return {"factor": s.a, "ipiv": s.ipiv, "x": s.b}
    if kind == "lu":
        s.a.copy_(s.a0)
        s.b.copy_(s.b0)
        s.check(s.zh.zmlhip_dgetrf(*s.factor))
        s.check(s.zh.zmlhip_dgetrs(*s.solve))
        return {"factor": s.a, "info": s.info, "ipiv": s.ipiv, "x": s.b}
    if kind == "chol":
        s.a.copy_(s.a0)
        s.b.copy_(s.b0)
        s.check(s.zh.zmlhip_dpotrf(*s.factor))
        s.check(s.zh.zmlhip_dpotrs(*s.solve))
        return {"factor": s.a, "info": s.info, "x": s.b}
    if kind == "batch":
        s.check(s.zh.zmlhip_batch_plan_execute(s.plan, s.stream))
        return s.x
    s.check(s.call(*s.args))
    return s.x


# ---- algorithmic work ---------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "gemv":
        m, n = case["m"], case["n"]
        return {"bytes": 8.0 * (m * n + m + n), "flops": 2.0 * m * n}
    if kind == "gemm":
        m, n, k, w = case["m"], case["n"], case["k"], 8.0 if case["dtype"] == "f64" else 4.0
        return {"bytes": w * (m * k + k * n + (1 if case["beta"] == 0.0 else 2) * m * n), "flops": 2.0 * m * n * k}
    if kind == "trsm":
        m, n = case["m"], case["n"]
        q = m if case["side"] == "L" else n
        return {"bytes": 8.0 * (q * q / 2 + 2 * m * n), "flops": 1.0 * q * m * n}
    if kind == "batch":
        w = {"bytes": 0.0, "flops": 0.0}
        for (n, nrhs, spd), ids in _batch_sizes(case):
            w["bytes"] += len(ids) * 8.0 * (n * n + 2 * n * nrhs)
            w["flops"] += len(ids) * ((1.0 if spd else 2.0) / 3.0 * n ** 3 + 2.0 * n * n * nrhs)
        return w
    n, nrhs = case["n"], case["nrhs"]
    if kind in ("lu", "gesv_host"):
        return {"bytes": 8.0 * (2 * n * n + 2 * n * nrhs), "flops": 2.0 / 3.0 * n ** 3 + 2.0 * n * n * nrhs}
    if kind == "chol":
        return {"bytes": 8.0 * (n * n + 2 * n * nrhs), "flops": n ** 3 / 3.0 + 2.0 * n * n * nrhs}
    # the solvers leave A as it is and return x alone
    third = 2.0 if kind == "mixed_lu" else 1.0
    return {"bytes": 8.0 * (n * n * third / 2 + 2 * n * nrhs), "flops": third / 3.0 * n ** 3 + 2.0 * n * n * nrhs}


# ---- the same in plain 64-bit torch --------------------------------------------------
def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        out = []
        for n, nrhs, _, _, A, B in _batch_inputs(case, seed):
            # column-major storage: the stored (row-major) matrix is A^T, the right-hand sides are rows
            out.append(torch.linalg.solve(A.transpose(1, 2).contiguous(), B.transpose(1, 2).contiguous())
                       .transpose(1, 2).reshape(-1))
        return torch.cat(out)
    ops = _inputs(case, seed)
    if kind == "gemv":
        A = ops[0] if case["trans"] == "N" else ops[0].t()
        return A @ ops[1] + case["beta"] * ops[2]
    if kind == "gemm":
        A, B, C = (t.double() for t in ops)
        A, B = A if case["ta"] == "N" else A.t(), B if case["tb"] == "N" else B.t()
        return _stored(A @ B + case["beta"] * C, case["layout"])[0]
    if kind == "trsm":
        A, B = ops
        upper = case["uplo"] == "U"
        A = (A.triu() if upper else A.tril())
        if case["trans"] == "T":
            A, upper = A.t(), not upper
        X = torch.linalg.solve_triangular(A.contiguous(), B, upper=upper, left=case["side"] == "L",
                                          unitriangular=case["diag"] == "U")
        return _stored(X, case["layout"])[0]
    if kind in ("lu", "gesv_host"):
        # on the host: the device library's factorization does not always take the largest pivot
        A, B = (t.cpu() for t in ops)
        LU, piv = torch.linalg.lu_factor(A)
        X = torch.linalg.lu_solve(LU, piv, B)
        out = {"factor": _stored(LU, case["layout"])[0], "ipiv": None, "x": _stored(X, case["layout"])[0]}
        if kind == "lu":
            out["info"] = None
        return out
    if kind == "chol":
        A, B = ops
        L = torch.linalg.cholesky(A)
        X = torch.cholesky_solve(B, L)
        F = L.tril() + A.triu(1) if case["uplo"] == "L" else L.tril().t() + A.tril(-1)
        return {"factor": _stored(F, case["layout"])[0], "info": None, "x": _stored(X, case["layout"])[0]}
    return _stored(ops[2], case["layout"])[0]   # the right-hand side was formed from it, in 64 bits
