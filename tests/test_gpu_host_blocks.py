"""Calls on host memory that follow each other on kept device blocks: growing and
shrinking sizes, blocks above and below the size that is kept, a call that ends
early (singular matrix, bad argument) in between, and several threads at once.
Every result has to be the bits of the same call made first."""
import threading

import numpy as np
import pytest

from tests.helpers import ROW, P

pytestmark = pytest.mark.gpu

SIZES = (200, 16, 350, 64, 1500, 201, 33)   # 1500: an 18 MB matrix, not kept


def gesv(zh, n, seed):
    rng = np.random.default_rng(seed)
    a, b, ip = rng.uniform(-1, 1, (n, n)), rng.uniform(-1, 1, (n, 2)), np.zeros(n, np.int32)
    assert zh.LAPACKE_dgesv(ROW, n, 2, P(a), n, P(ip), P(b), 2) == 0
    return a, b, ip


def test_results_do_not_depend_on_earlier_calls(zh, torch_cuda):
    first = {n: gesv(zh, n, n) for n in SIZES}
    for n in reversed(SIZES):
        a, ip = np.ones((40, 40)), np.zeros(40, np.int32)
        b = np.ones((40, 1))
        assert zh.LAPACKE_dgesv(ROW, 40, 1, P(a), 40, P(ip), P(b), 1) > 0      # singular
        assert zh.LAPACKE_dgesv(ROW, 40, 1, P(a), 39, P(ip), P(b), 1) == -5
        for got, want in zip(gesv(zh, n, n), first[n]):
            assert np.array_equal(got, want)


def test_threads_have_their_own_blocks(zh, torch_cuda):
    want = {n: gesv(zh, n, n) for n in SIZES}
    wrong = []

    def work(k):
        for n in SIZES[k:] + SIZES[:k]:
            if not all(np.array_equal(g, w) for g, w in zip(gesv(zh, n, n), want[n])):
                wrong.append((k, n))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
