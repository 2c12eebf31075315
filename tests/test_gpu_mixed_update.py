"""The low-precision trailing update at orders whose updates write C past the
caches (an update of more than 256 MB) and at ragged ones: the block rows and
columns at the edge of C, whole tiles inside it, and the lower triangle only.

A wrong entry of an update spoils the factors, so that the refinement no longer
converges in the few steps which the precision of the operands gives: with
operands of 11 (8) bits and the growth of these diagonally heavy matrices each
step gains more than 2 (1) digits, so 8 steps without GMRES or the FP64
factorization are a bound with room. The solution has to meet the bar of the
other mixed solves, a normwise backward error of at most 16 n u.
"""
import ctypes

import pytest

from tests.helpers import COL, ROW, P

pytestmark = pytest.mark.gpu


def solve(zh, torch, call, A, B, precision):
    from zml_amd._lib import IROpts, IRResult
    n, nrhs = B.shape
    X = torch.zeros_like(B)
    r = IRResult()
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    rc = call(n, nrhs, P(A), P(B), P(X), ctypes.byref(IROpts(precision=precision)), ctypes.byref(r), s)
    assert rc == 0, (rc, zh.zmlhip_last_error())
    torch.cuda.synchronize()
    be = ((B - A @ X).abs().amax(0) / X.abs().amax(0)).max() / A.abs().sum(1).max() / (n * 2.0 ** -53)
    assert r.info == 0 and r.fallback == 0 and r.gmres_iterations == 0
    assert r.iterations <= 8
    assert float(be) <= 16


@pytest.mark.parametrize("precision,n", [(1, 8840), (2, 8840), (1, 8704), (1, 1609), (2, 1609), (1, 1664)])
def test_lu_update(zh, torch_cuda, precision, n):
    torch = torch_cuda
    g = torch.Generator(device="cuda")
    g.manual_seed(n + precision)
    A = torch.rand(n, n, dtype=torch.float64, device="cuda", generator=g).sub_(0.5)
    A.diagonal().add_(0.1 * n)
    B = torch.rand(n, 1, dtype=torch.float64, device="cuda", generator=g)
    solve(zh, torch, lambda n, k, a, b, x, o, r, s: zh.zmlhip_dgesv_mixed(ROW, n, k, a, n, b, k, x, k, o, r, s),
          A, B, precision)


@pytest.mark.parametrize("precision,n", [(1, 12333), (1, 1609), (2, 1609)])
def test_cholesky_update(zh, torch_cuda, precision, n):
    torch = torch_cuda
    g = torch.Generator(device="cuda")
    g.manual_seed(n + precision)
    A = torch.rand(n, n, dtype=torch.float64, device="cuda", generator=g).sub_(0.5)
    A = A + A.t()
    A.diagonal().add_(0.1 * n)      # the off-diagonal part has norm about sqrt(n / 1.5)
    B = torch.rand(n, 2, dtype=torch.float64, device="cuda", generator=g)
    solve(zh, torch, lambda n, k, a, b, x, o, r, s: zh.zmlhip_dposv_mixed(ROW, b"L", n, k, a, n, b, k, x, k, o, r, s),
          A, B, precision)


@pytest.mark.parametrize("n,ties", [(512, False), (1324, False), (1324, True)])
def test_diagonal_block_pivots(zh, torch_cuda, n, ties):
    """Pivots from every row of the 256-row diagonal blocks: the rows of a
    diagonally heavy matrix in random order inside each block (with `ties`, equal
    entries off the diagonal, so that a column's candidates tie until the pivots
    of earlier ones tell them apart). Every block column must go through."""
    from zml_amd._lib import IROpts, IRResult
    torch = torch_cuda
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    A = torch.full((n, n), 0.25, dtype=torch.float64, device="cuda") if ties else \
        torch.rand(n, n, dtype=torch.float64, device="cuda", generator=g).sub_(0.5)
    A.diagonal().add_(0.1 * n)
    p = torch.cat([k + torch.randperm(min(256, n - k), generator=g, device="cuda") for k in range(0, n, 256)])
    A = A[p].contiguous()
    B = torch.rand(n, 1, dtype=torch.float64, device="cuda", generator=g)
    X, r = torch.zeros_like(B), IRResult()
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    rc = zh.zmlhip_dgesv_mixed(ROW, n, 1, P(A), n, P(B), 1, P(X), 1, ctypes.byref(IROpts(precision=0)),
                               ctypes.byref(r), s)
    assert rc == 0, (rc, zh.zmlhip_last_error())
    torch.cuda.synchronize()
    be = float((B - A @ X).abs().max() / X.abs().max() / A.abs().sum(1).max() / (n * 2.0 ** -53))
    assert r.info == 0 and r.fallback == 0 and r.gmres_iterations == 0 and r.iterations <= 3
    assert r.panels == n // 512 and r.panels_optimistic == r.panels
    assert be <= 16
