"""Triangular solves whose values leave the range of the fast substitution (NaN,
infinities, magnitudes near the ends of the range, zeros on the diagonal): within
one 64-row block the results are the bits of the plain substitution, with
separately rounded products and differences, and such a solve costs a small
multiple of an ordinary one."""
import ctypes

import numpy as np
import pytest

from tests.helpers import COL, P, store

pytestmark = pytest.mark.gpu

KINDS = ["plain", "nan", "inf", "tiny", "huge", "mixed", "zero_pivot", "subnormal"]


def substitution(M, B, mode):
    X = B.copy()
    for k in range(len(M)):
        if mode == "div":
            X[k] = X[k] / M[k, k]
        elif mode == "mul":
            X[k] = X[k] * (M.dtype.type(1) / M[k, k])
        for r in range(k + 1, len(M)):
            X[r] = X[r] - X[k] * M[r, k]
    return X


def system(kind, q, nvec, dtype, rng):
    big = 200 if dtype == np.float64 else 30
    M = np.tril(rng.uniform(-1, 1, (q, q)) / np.sqrt(q)) + np.diag(rng.uniform(1, 2, q))
    B = rng.uniform(-1, 1, (q, nvec))
    if kind == "nan":
        B[q // 2, 0] = np.nan
    elif kind == "inf":
        B[q // 3, nvec // 2] = -np.inf
    elif kind == "tiny":
        B *= 10.0 ** -big
    elif kind == "huge":
        M *= 10.0 ** big
        B *= 10.0 ** big
    elif kind == "mixed":       # each vector in another part of the range
        B *= 10.0 ** rng.integers(-big, big, nvec)
    elif kind == "zero_pivot":
        M[q // 2, q // 2] = 0.0
    elif kind == "subnormal":
        B *= float(np.finfo(dtype).tiny)
    return M.astype(dtype), B.astype(dtype)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("mode", ["div", "mul", "unit"])
@pytest.mark.parametrize("q", [1, 2, 7, 8, 9, 15, 16, 17, 32, 33, 48, 49, 63, 64])
def test_bits_of_the_plain_substitution(zh, kind, dtype, mode, q):
    nvec = 21
    rng = np.random.default_rng(q + 100 * KINDS.index(kind))
    M, B = system(kind, q, nvec, dtype, rng)
    with np.errstate(all="ignore"):
        want = substitution(M, B, mode)
    trsm = zh.cblas_dtrsm if dtype == np.float64 else zh.cblas_strsm
    diag = 132 if mode == "unit" else 131
    a = store(COL, M, q).astype(dtype)
    if mode == "mul":           # X op(A) = B with A = M^T upper: the vectors are rows
        a, b = store(COL, M.T, q).astype(dtype), store(COL, B.T, nvec).astype(dtype)
        trsm(COL, 142, 121, 111, diag, nvec, q, 1.0, P(a), q, P(b), nvec)
        got = b.reshape(q, nvec)
    else:
        b = store(COL, B, q).astype(dtype)
        trsm(COL, 141, 122, 111, diag, q, nvec, 1.0, P(a), q, P(b), q)
        got = b.reshape(nvec, q).T
    assert np.array_equal(got, want, equal_nan=True)


@pytest.mark.parametrize("kind", ["nan", "tiny", "huge"])
def test_cost_outside_the_fast_range(zh, torch_cuda, kind):
    """512 rows, 16 vectors, all of them outside. A masked step with an exact quotient
    is a chain of three to four times the fast one's length, beside sums that cost the
    same: 5 times the ordinary solve is a bound with room."""
    torch = torch_cuda
    q, nvec = 512, 16
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def time_of(kind):
        M, B = system(kind, q, nvec, np.float64, np.random.default_rng(1))
        if kind == "nan":
            B[0] = np.nan
        a, b0 = torch.from_numpy(np.ascontiguousarray(M.T)).cuda(), torch.from_numpy(np.ascontiguousarray(B.T)).cuda()
        best = float("inf")
        for _ in range(10):
            b = b0.clone()
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            assert zh.zmlhip_dtrsm(COL, 141, 122, 111, 131, q, nvec, 1.0, P(a), q, P(b), q, s) == 0
            e1.record()
            torch.cuda.synchronize()
            best = min(best, e0.elapsed_time(e1))
        return best

    assert time_of(kind) <= 5 * time_of("plain")
