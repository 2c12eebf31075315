"""The batched solver's accumulator-tile kernels (64 < n <= 256): orders at the
edges of its 16-column chunks, 32-row tiles and 64-row lanes, and right-hand
sides at the edges of the groups of four that are refined together.

Held to the other batched tests' bars: backward error at most 16 n u, and for
these well-conditioned systems 1e-12 of the oracle's solution.
"""
import numpy as np
import pytest

from tests.test_gpu_batched import Batch, check

pytestmark = pytest.mark.gpu

ORDERS = [65, 79, 80, 81, 95, 96, 97, 112, 127, 128, 129, 143, 144, 145, 160, 161, 191, 192, 193, 224, 241, 255, 256]


def system(rng, n, nrhs, spd):
    A = rng.uniform(-1, 1, (n, n))
    if spd:
        A = A @ A.T / n + np.eye(n)
    else:
        A = (A + n / 4.0 * np.eye(n))[rng.permutation(n)]   # pivots from every row
    return A, rng.uniform(-1, 1, (n, nrhs)), spd


@pytest.mark.parametrize("spd", [False, True])
def test_orders_and_groups(zh, torch_cuda, spd):
    rng = np.random.default_rng(31 + spd)
    systems = [system(rng, n, 1 + i % 9, spd) for i, n in enumerate(ORDERS)]
    bt = Batch(zh, torch_cuda, systems, autotune=0)
    status, hx = bt.run()
    check(bt, status, hx)
    status2, hx2 = bt.run()
    assert np.array_equal(status, status2) and np.array_equal(hx, hx2)
    bt.close()


def test_singular_and_nan_systems_fail_alone(zh, torch_cuda):
    rng = np.random.default_rng(5)
    good = [system(rng, n, 5, False) for n in (70, 130, 256)]
    A0, B0, _ = system(rng, 150, 2, False)
    A0[:, 37] = 0.0
    A1, B1, _ = system(rng, 90, 2, False)
    A1[3, 5] = np.nan
    systems = [good[0], (A0, B0, False), good[1], (A1, B1, False), good[2]]
    bt = Batch(zh, torch_cuda, systems, autotune=0)
    status, hx = bt.run()
    bt.close()
    assert status[1] == -1 and status[3] == -1
    solved = list(bt.solutions(hx))
    for i in (0, 2, 4):
        A, Bv, _ = systems[i]
        assert status[i] >= 0
        an = np.abs(A).sum(1).max()
        for q in range(Bv.shape[1]):
            x = solved[i][:, q]
            assert np.abs(Bv[:, q] - A @ x).max() / (an * np.abs(x).max() * A.shape[0] * 2.0 ** -53) <= 16
