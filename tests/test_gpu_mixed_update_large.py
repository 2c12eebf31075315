"""Low-precision trailing updates that write C past the caches, at orders that are
no multiple of the tile: the block rows and columns at the edge of C (the buffer
descriptor's end, columns sent past it, partial rows of scales), whole tiles, and
the lower triangle only. The bounds are those of the smaller updates' tests."""
import os
import re

import pytest

from tests.helpers import ROW, P
from tests.test_gpu_mixed_update import solve

pytestmark = pytest.mark.gpu

SOURCE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "zml_amd", "csrc", "mp_gemm.hip")


def past_the_caches(tiles):
    mib = int(re.search(r"if \(tiles \* \(MT \* NTL \* 4\) > \(int64_t\((\d+)\) << 20\)\)", open(SOURCE).read()).group(1))
    return tiles * 128 * 128 * 4 > mib << 20


def up(x):
    return -(-x // 128)


@pytest.mark.parametrize("precision,n", [(1, 9233), (2, 9233), (1, 9200), (1, 9217), (1, 9343), (1, 9344)])
def test_lu(zh, torch_cuda, precision, n):
    # the first update: all rows below the block column, without the next 512 columns
    assert past_the_caches(up(n - 512) * up(n - 1024))
    torch = torch_cuda
    g = torch.Generator(device="cuda")
    g.manual_seed(n + precision)
    A = torch.rand(n, n, dtype=torch.float64, device="cuda", generator=g).sub_(0.5)
    A.diagonal().add_(0.1 * n)
    B = torch.rand(n, 1, dtype=torch.float64, device="cuda", generator=g)
    solve(zh, torch, lambda n, k, a, b, x, o, r, s: zh.zmlhip_dgesv_mixed(ROW, n, k, a, n, b, k, x, k, o, r, s),
          A, B, precision)


@pytest.mark.parametrize("precision,n", [(1, 12653), (2, 12653), (1, 12800)])
def test_cholesky(zh, torch_cuda, precision, n):
    t = up(n - 1024)
    assert past_the_caches(t * (t + 1) // 2)
    torch = torch_cuda
    g = torch.Generator(device="cuda")
    g.manual_seed(n + precision)
    A = torch.rand(n, n, dtype=torch.float64, device="cuda", generator=g).sub_(0.5)
    A = A + A.t()
    A.diagonal().add_(0.1 * n)
    B = torch.rand(n, 2, dtype=torch.float64, device="cuda", generator=g)
    solve(zh, torch, lambda n, k, a, b, x, o, r, s: zh.zmlhip_dposv_mixed(ROW, b"L", n, k, a, n, b, k, x, k, o, r, s),
          A, B, precision)
