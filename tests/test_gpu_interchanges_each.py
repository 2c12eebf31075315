"""Row interchanges around the lines between composed moves and one thread per
column (few interchanges, many columns), both storage orders and directions,
with entries of ipiv that name no row. Moves are exact."""
import ctypes

import numpy as np
import pytest

from tests.helpers import COL, ROW, P

pytestmark = pytest.mark.gpu


def swap(zh, torch, order, a, n, ld, k1, k2, dp, incx):
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert zh.zmlhip_dlaswp(order, n, P(a), ld, k1, k2, P(dp), incx, s) == 0


@pytest.mark.parametrize("order", [ROW, COL])
@pytest.mark.parametrize("incx", [1, -1, 2])
@pytest.mark.parametrize("steps,n", [(1, 1), (8, 5), (8, 300), (9, 5), (9, 575), (9, 576), (9, 6299), (9, 6300),
                                     (256, 4999), (256, 5000), (257, 5000), (257, 14000)])
def test_lines_of_the_dispatch(zh, torch_cuda, order, incx, steps, n):
    torch = torch_cuda
    m, k1 = steps + 40, 3
    rng = np.random.default_rng(steps + n + order + incx)
    ip = rng.integers(1, m + 1, steps).astype(np.int32)
    ip[1::7] = 0
    ipiv = np.zeros(k1 - 1 + (steps - 1) * abs(incx) + 1, np.int32)
    ipiv[k1 - 1::abs(incx)] = ip
    A = rng.uniform(-1, 1, (m, n))
    want = A.copy()
    for e in range(steps) if incx > 0 else range(steps - 1, -1, -1):
        if ip[e] >= 1:
            i, j = k1 - 1 + e, ip[e] - 1
            want[[i, j]] = want[[j, i]]
    ld = (n if order == ROW else m) + 1
    buf = np.zeros((m, ld) if order == ROW else (n, ld))
    buf[:, :ld - 1] = A if order == ROW else A.T
    a = torch.from_numpy(buf).cuda()
    swap(zh, torch, order, a, n, ld, k1, k1 + steps - 1, torch.from_numpy(ipiv).cuda(), incx)
    torch.cuda.synchronize()
    got = a.cpu().numpy()
    assert np.array_equal(got[:, ld - 1], buf[:, ld - 1])
    assert np.array_equal(got[:, :-1] if order == ROW else got[:, :-1].T, want)


@pytest.mark.parametrize("steps", [4, 16])
def test_many_columns_cost_their_memory_traffic(zh, torch_cuda, steps):
    """Along rows, 100,000 columns: 3 (13) MB read and written, a few microseconds
    beside the call's own twelve: three times the call on 64 columns is a bound with room."""
    torch = torch_cuda
    n = 100000
    a = torch.rand(100, n, dtype=torch.float64, device="cuda")
    dp = torch.arange(steps + 1, 2 * steps + 1, dtype=torch.int32, device="cuda")

    def time_of(cols):
        best = float("inf")
        for _ in range(20):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            swap(zh, torch, ROW, a, cols, n, 1, steps, dp, 1)
            e1.record()
            torch.cuda.synchronize()
            best = min(best, e0.elapsed_time(e1))
        return best

    assert time_of(n) <= 3 * time_of(64)
