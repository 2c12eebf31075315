"""The one-workgroup Cholesky of a diagonal block (orders up to 128, chunks of 16
columns): lower, column-major factors equal the oracle's bit for bit (every
element receives the same separately rounded operations in the same order), at
the edges of the chunks, near the ends of the exponent range and up to a failing
pivot."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import COL, P, dense, store

pytestmark = pytest.mark.gpu


def _spd(n, seed, exponents=0):
    rng = np.random.default_rng(seed)
    B = rng.uniform(-1, 1, (n, n))
    A = B @ B.T / n + np.eye(n)
    A = np.tril(A) + np.tril(A, -1).T
    if exponents:   # D A D with powers of two keeps it SPD and every rounding the same
        d = rng.integers(-exponents, exponents, n)
        A = np.ldexp(np.ldexp(A, d[:, None]), d[None, :])
    return A


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 33, 64, 100, 112, 113, 127, 128])
@pytest.mark.parametrize("exponents", [0, 300])
def test_diagonal_block_bits(zh, n, exponents):
    A = _spd(n, n, exponents)
    a, ref = store(COL, A, n + 1), store(COL, A, n + 1)
    assert O.potrf(COL, 122, n, ref, n + 1) == 0
    assert zh.LAPACKE_dpotrf(COL, b"L", n, P(a), n + 1) == 0
    assert np.array_equal(np.tril(dense(COL, n, n, a, n + 1)), np.tril(dense(COL, n, n, ref, n + 1)))
    u = store(COL, A, n)   # upper: the same values transposed
    assert zh.LAPACKE_dpotrf(COL, b"U", n, P(u), n) == 0
    assert np.array_equal(np.triu(dense(COL, n, n, u, n)).T, np.tril(dense(COL, n, n, ref, n + 1)))


@pytest.mark.parametrize("k", [0, 1, 15, 16, 47, 48, 63, 64, 65, 126, 127])
@pytest.mark.parametrize("value", [-1.0, 0.0, np.nan])
def test_failing_pivot(zh, k, value):
    n = 128
    A = _spd(n, 7)
    ref = store(COL, A, n)
    assert O.potrf(COL, 122, n, ref, n) == 0
    A[k, k] = value if value != 0.0 or k == 0 else -1e-3
    a = store(COL, A, n)
    assert zh.LAPACKE_dpotrf(COL, b"L", n, P(a), n) == k + 1
    got, L = dense(COL, n, n, a, n), dense(COL, n, n, ref, n)
    lead = np.tril(L)[:k, :k]
    assert np.array_equal(np.tril(got)[:k, :k], lead)   # the columns before it are final


def test_square_roots_and_reciprocals(zh):
    """2 x 2 blocks [[d, .], [x, 4]]: l11 = sqrt(d) and l21 = fl(x fl(1 / l11)), correctly rounded."""
    rng = np.random.default_rng(5)
    d = np.concatenate([np.ldexp(rng.uniform(1, 4, 60), 2 * rng.integers(-254, 254, 60)),
                        np.ldexp(rng.uniform(1, 2, 20), rng.integers(-1000, -514, 20)),
                        np.nextafter(np.ldexp(1.0, rng.integers(-500, 500, 20)), 0.0)])
    for v in d:
        x = np.sqrt(v) * rng.uniform(0.1, 0.9)
        a = np.array([v, x, 0.0, 4.0])   # l21 < 1: positive definite
        assert zh.LAPACKE_dpotrf(COL, b"L", 2, P(a), 2) == 0
        l = np.sqrt(v)
        assert a[0] == l and a[1] == x * (1.0 / l)
