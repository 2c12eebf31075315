"""Row interchanges through composed moves (dlaswp, and the LU's block columns
through getrf): pivots in LAPACK's form and arbitrary ones, chains that hand one
row through all the others, repeated rows, both directions, and lists around the
256 interchanges that are composed at a time. Moves are exact."""
import ctypes

import numpy as np
import pytest

from tests.helpers import COL, ROW, P, dense, store

pytestmark = pytest.mark.gpu


def pivots(kind, m, rng):
    k = np.arange(1, m + 1)
    if kind == "lapack":
        return rng.integers(k, m + 1)
    if kind == "any":
        return rng.integers(1, m + 1, m)
    if kind == "chain":
        return np.minimum(k + 1, m)
    return np.full(m, m)   # "last": every row with the last one


@pytest.mark.parametrize("kind", ["lapack", "any", "chain", "last"])
@pytest.mark.parametrize("order", [ROW, COL])
@pytest.mark.parametrize("m,n,k1,k2,incx", [(40, 1, 1, 1, 1), (300, 7, 1, 256, 1), (300, 8, 3, 259, -1),
                                            (700, 9, 1, 700, 2), (1500, 17, 1, 1500, -1), (1500, 1, 2, 1400, -2)])
def test_dlaswp(zh, torch_cuda, kind, order, m, n, k1, k2, incx):
    torch = torch_cuda
    rng = np.random.default_rng(m + n + len(kind))
    A = rng.uniform(-1, 1, (m, n))
    ip = pivots(kind, m, rng).astype(np.int32)
    step = abs(incx)
    ipiv = np.zeros(k1 - 1 + (k2 - k1) * step + 1, np.int32)   # entry of row k (1-based) at k1 - 1 + (k - k1) |incx|
    ipiv[k1 - 1::step] = ip[k1 - 1:k2]
    want = A.copy()
    rows = range(k1 - 1, k2) if incx > 0 else range(k2 - 1, k1 - 2, -1)
    for i in rows:
        j = ip[i] - 1
        want[[i, j]] = want[[j, i]]
    ld = (m if order == COL else n) + 2
    a = torch.from_numpy(store(order, A, ld)).cuda()
    dp = torch.from_numpy(ipiv).cuda()
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert zh.zmlhip_dlaswp(order, n, P(a), ld, k1, k2, P(dp), incx, s) == 0
    torch.cuda.synchronize()
    assert np.array_equal(dense(order, m, n, a.cpu().numpy(), ld), want)


@pytest.mark.parametrize("n", [200, 256, 257, 520, 1100])
def test_getrf_block_columns_use_the_composed_moves(zh, torch_cuda, n):
    """P A = L U to rounding with every row displaced: a wrong move would be an error of order one."""
    torch = torch_cuda
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    A = torch.rand(n, n, dtype=torch.float64, device="cuda", generator=g).sub_(0.5)
    A = A[torch.randperm(n, generator=g, device="cuda")].contiguous()
    F, ip, info = A.clone(), torch.zeros(n, dtype=torch.int32, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert zh.zmlhip_dgetrf(ROW, n, n, P(F), n, P(ip), P(info), s) == 0
    torch.cuda.synchronize()
    assert int(info) == 0
    PA = A.clone().cpu()
    for k, p in enumerate(ip.cpu().tolist()):
        PA[[k, p - 1]] = PA[[p - 1, k]]
    L, U = F.tril(-1) + torch.eye(n, dtype=torch.float64, device="cuda"), F.triu()
    # |P A - L U| <= n u |L| |U| entry by entry
    err = (PA.cuda() - L @ U).abs()
    assert bool((err <= n * 2.0 ** -53 * (L.abs() @ U.abs())).all())
