"""The LU leaf (groups of 8 columns, virtual interchanges; one workgroup up to 512
rows, exchanging workgroups above) against the oracle bit for bit: a single leaf
(n <= 64 columns) has no matrix-core update in it, so factors, pivots and info equal zml's
exactly, at the edges of its row ranges and column groups, with exact ties, zero
columns, subnormal pivots, infinities and NaN."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import COL, P, ROW, dense, store

pytestmark = pytest.mark.gpu

ROWS = [1, 2, 63, 64, 65, 200, 256, 257, 511, 512, 513, 777, 1024, 1025]


def _matrix(kind, m, n, seed):
    rng = np.random.default_rng(seed)
    if kind == "ties":
        return rng.integers(-3, 4, (m, n)).astype(np.float64)
    a = rng.uniform(-1, 1, (m, n))
    if kind == "zero_column":
        a[:, n // 2] = 0.0
    elif kind == "subnormal":
        a[:, 0] = np.ldexp(a[:, 0], -1030)
    elif kind == "inf":
        a[m // 2, n // 3] = np.inf
    elif kind == "nan":
        a[m // 2, n // 3] = np.nan
    elif kind == "nan_first":
        a[0, 0] = np.nan
    return a


def _same(x, y):
    return np.array_equal(x, y, equal_nan=True)


@pytest.mark.parametrize("m", ROWS)
@pytest.mark.parametrize("n", [1, 7, 8, 9, 31, 32, 33, 40, 57, 64])
def test_dgetrf_one_leaf_bits(zh, m, n):
    order = ROW if (m + n) % 2 else COL
    for kind in ("uniform", "ties"):
        A = _matrix(kind, m, n, 7 * m + n)
        ld = (m if order == COL else n) + (m % 3)
        a, ref = store(order, A, ld), store(order, A, ld)
        ip, ip_ref = np.zeros(min(m, n), np.int32), np.zeros(min(m, n), np.int32)
        info_ref = O.getrf(order, m, n, ref, ld, ip_ref)
        assert zh.LAPACKE_dgetrf(order, m, n, P(a), ld, P(ip)) == info_ref
        assert np.array_equal(ip, ip_ref)
        k = min(m, n)   # columns beyond a square block go through the matrix cores
        assert _same(dense(order, m, n, a, ld)[:, :k], dense(order, m, n, ref, ld)[:, :k])


@pytest.mark.parametrize("m", [64, 200, 512, 1000])
@pytest.mark.parametrize("kind", ["zero_column", "subnormal", "inf", "nan", "nan_first"])
def test_dgetrf_one_leaf_special_values(zh, m, kind):
    n = 48
    A = _matrix(kind, m, n, m)
    a, ref = store(ROW, A, n), store(ROW, A, n)
    ip, ip_ref = np.zeros(n, np.int32), np.zeros(n, np.int32)
    info_ref = O.getrf(ROW, m, n, ref, n, ip_ref)
    assert zh.LAPACKE_dgetrf(ROW, m, n, P(a), n, P(ip)) == info_ref
    assert np.array_equal(ip, ip_ref)
    assert _same(dense(ROW, m, n, a, n), dense(ROW, m, n, ref, n))


@pytest.mark.parametrize("m", ROWS)
def test_sgetrf_one_leaf_bits(zh, m):
    n = min(m, 50)
    A = _matrix("uniform", m, n, m).astype(np.float32)
    a, ref = A.reshape(-1).copy(), A.reshape(-1).copy()
    ip, ip_ref = np.zeros(n, np.int32), np.zeros(n, np.int32)
    assert O.sgetrf(ROW, m, n, ref, n, ip_ref) == zh.LAPACKE_sgetrf(ROW, m, n, P(a), n, P(ip))
    assert np.array_equal(ip, ip_ref)
    assert np.array_equal(a, ref)
