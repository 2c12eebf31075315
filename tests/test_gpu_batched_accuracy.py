"""How far the batched solver's solutions are from the exact ones, and what it says of
systems that it cannot solve.

Refinement ends with x = fl(x + d), d from the residual as FP64 arithmetic gives it:
what is left in the error is the rounding of that residual, so its sums decide.
The kernels sum in parts (of 8 columns, or of interleaved ones); a sum over one
column after the other onto b leaves errors about twice as large."""
import numpy as np
import pytest

from tests.test_gpu_batched import Batch

COUNT, NRHS = 60, 2


def systems(n, seed):
    rng = np.random.default_rng(seed)
    return rng.uniform(-1, 1, (COUNT, n, n)) + n / 4.0 * np.eye(n), rng.uniform(-1, 1, (COUNT, n, NRHS))


def exact(A, B):
    """The solutions to well below u, from refinement in extended precision."""
    L, X = A.astype(np.longdouble), np.linalg.solve(A, B).astype(np.longdouble)
    for _ in range(3):
        R = B.astype(np.longdouble) - np.stack([a @ x for a, x in zip(L, X)])
        X = X + np.linalg.solve(A, R.astype(np.float64))
    return X


def refined(A, B, part):
    """Three refinement steps with an FP32 inverse and residuals summed in parts of
    `part` columns (0: one after the other onto b)."""
    inv = np.linalg.inv(A.astype(np.float32))
    X = np.zeros_like(B)
    n = A.shape[1]
    for step in range(3):
        R = B.copy()
        if step:
            total, acc = np.zeros_like(B), np.zeros_like(B)
            for j in range(n):
                p = A[:, :, j, None] * X[:, None, j, :]
                if part == 0:
                    R = R - p
                    continue
                acc = acc + p
                if j % part == part - 1 or j == n - 1:
                    total, acc = total + acc, np.zeros_like(B)
            R = R - total
        X = X + np.matmul(inv, R.astype(np.float32)).astype(np.float64)
    return X


def mean_error(X, E):
    e = np.abs(X - E).max(axis=1) / np.abs(E).max(axis=1)
    return float(np.exp(np.log(e.astype(np.float64)).mean()))


def test_the_order_of_the_sums_shows():
    A, B = systems(128, 1)
    E = exact(A, B)
    assert mean_error(refined(A, B, 0), E) > 1.25 * mean_error(refined(A, B, 8), E)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [70, 100, 128, 130, 200, 256])
def test_errors_of_residuals_summed_in_parts(zh, torch_cuda, n):
    """120 solutions: the mean of their errors' logarithms has a standard deviation of a
    few hundredths, so 1.15 times the reference's mean is three or more of them away."""
    A, B = systems(n, n)
    bt = Batch(zh, torch_cuda, [(a, b, False) for a, b in zip(A, B)], autotune=0)
    status, hx = bt.run()
    X = np.stack(list(bt.solutions(hx)))
    bt.close()
    assert np.all(status >= 0)
    E = exact(A, B)
    assert mean_error(X, E) <= 1.15 * mean_error(refined(A, B, 8), E)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [20, 40, 70, 110, 128, 150, 200, 256])
@pytest.mark.parametrize("decades", [20, 25, 30, 35])
def test_no_success_without_a_solution(zh, torch_cuda, n, decades):
    """Columns over up to 70 decades, which the FP32 factors cannot hold: some entries of
    a solution come out as NaN while others are numbers. Such a system has to say so."""
    rng = np.random.default_rng(n + decades)
    c = 10.0 ** rng.uniform(-decades, decades, (20, n))
    A = (rng.uniform(-1, 1, (20, n, n)) + n / 4.0 * np.eye(n)) * c[:, None, :]
    B = np.matmul(A, rng.uniform(-1, 1, (20, n, 2)) / c[:, :, None])
    bt = Batch(zh, torch_cuda, [(a, b, False) for a, b in zip(A, B)], autotune=0)
    status, hx = bt.run()
    for k, X in enumerate(bt.solutions(hx)):
        if status[k] >= 0:
            R = np.abs(B[k] - A[k] @ X).max(axis=0)
            assert np.all(R <= 16 * n * 2.0 ** -53 * np.abs(A[k]).sum(1).max() * np.abs(X).max(axis=0))
    bt.close()
