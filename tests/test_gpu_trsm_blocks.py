"""The blocked triangular solve at the edges of its blocks (64-row triangles,
512-row strips, 16-vector tiles, the 64-vector limit of the update for few
vectors), in every side / uplo / trans / diag form, and with values that leave
the fast substitution: zeros on the diagonal, infinities, NaN and magnitudes
near the ends of the range."""
import numpy as np
import pytest
from scipy.linalg import solve_triangular

from tests.helpers import COL, P, ROW, dense, store

pytestmark = pytest.mark.gpu


def _tri(q, seed):
    rng = np.random.default_rng(seed)
    return rng.uniform(-1, 1, (q, q)) / np.sqrt(q) + np.diag(rng.uniform(1, 2, q))


@pytest.mark.parametrize("side,uplo", [(141, 121), (141, 122), (142, 121), (142, 122)])
@pytest.mark.parametrize("trans", [111, 112])
@pytest.mark.parametrize("q,nvec", [(1, 1), (63, 16), (64, 17), (65, 1), (512, 33), (513, 64), (576, 65), (1090, 15),
                                    (1100, 129)])
def test_trsm_block_edges(zh, side, uplo, trans, q, nvec):
    order = ROW if (q + nvec) % 2 else COL
    diag = 132 if (q + uplo + trans) % 3 == 0 else 131
    T = _tri(q, q + nvec + side + uplo + trans)
    m, n = (q, nvec) if side == 141 else (nvec, q)
    B = np.random.default_rng(q).uniform(-1, 1, (m, n))
    lda, ldb = q + 3, (m if order == COL else n) + 1
    a, b = store(order, T, lda), store(order, B, ldb)
    zh.cblas_dtrsm(order, side, uplo, trans, diag, m, n, 1.0, P(a), lda, P(b), ldb)
    got = dense(order, m, n, b, ldb)
    lower = uplo == 122
    kw = dict(lower=lower, trans=0 if trans == 111 else 1, unit_diagonal=diag == 132)
    if side == 141:
        ref = solve_triangular(T, B, **kw)
    else:   # X op(T) = B  <=>  op(T)^T X^T = B^T
        ref = solve_triangular(T, B.T, **{**kw, "trans": 1 - kw["trans"]}).T
    # both are backward stable: |got - ref| <= 2 q u cond(op(T)) |ref|, cond below 50 for these triangles
    assert np.abs(got - ref).max() <= 2 * q * 2.0 ** -53 * 50 * max(np.abs(ref).max(), 1.0)


@pytest.mark.parametrize("trans", [111, 112])
def test_trsm_values_outside_the_fast_path(zh, trans):
    q, nvec = 130, 5
    lower = trans == 111                       # op(T) lower: solved from row 0 down
    T = np.tril(_tri(q, 3)) if lower else np.triu(_tri(q, 3))
    uplo = 122 if lower else 121
    B = np.random.default_rng(4).uniform(-1, 1, (q, nvec))
    op = T if lower else T.T

    def solve(Tm, Bm):
        a, b = store(COL, Tm, q), store(COL, Bm, q)
        zh.cblas_dtrsm(COL, 141, uplo, trans, 131, q, nvec, 1.0, P(a), q, P(b), q)
        return dense(COL, q, nvec, b, q)

    ref = solve_triangular(op, B, lower=True)
    # a zero pivot, an infinity, a NaN: rows solved before it keep their values
    for row, plant in ((70, "zero"), (33, "inf"), (129, "nan")):
        T2, B2 = T.copy(), B.copy()
        if plant == "zero":
            T2[row, row] = 0.0
        else:
            B2[row, 2] = np.inf if plant == "inf" else np.nan
        got = solve(T2, B2)
        assert np.array_equal(got[:row], solve(T, B)[:row])
        assert np.abs(got[:row] - ref[:row]).max() <= 1e-12
        assert not np.isfinite(got[row, 2])
    # scaling every row of the system by a power of two changes no quotient: the
    # solution is the same bit for bit, also where the corrected reciprocal would leave its range
    base = solve(T, B)
    for e in (-600, 700):
        assert np.array_equal(solve(np.ldexp(T, e), np.ldexp(B, e)), base)
