"""GEMM at the edges of its 64 x 64 tiles and 16-wide k-slabs, where k is split
over workgroups (few tiles, long k) and around the change to 128 x 128 tiles, in
every transpose form, FP64 and FP32, against a product in higher precision."""
import numpy as np
import pytest

from tests.helpers import COL, P, ROW, dense, store

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (64, 64, 16), (63, 65, 15), (65, 63, 17), (1, 130, 129), (128, 1, 255), (100, 90, 256),
          (33, 70, 600), (64, 64, 4100), (200, 10, 1111), (129, 129, 128)]


@pytest.mark.parametrize("order", [ROW, COL])
@pytest.mark.parametrize("ta,tb", [(111, 111), (112, 111), (111, 112), (112, 112)])
@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_gemm_edges(zh, order, ta, tb, m, n, k, dtype):
    rng = np.random.default_rng(m + 7 * n + 13 * k + ta + 3 * tb)
    alpha, beta = [(1.0, 0.0), (-1.0, 1.0), (0.5, 0.25)][(m + n + k) % 3]
    A = rng.uniform(-1, 1, (m, k)).astype(dtype)
    B = rng.uniform(-1, 1, (k, n)).astype(dtype)
    C = rng.uniform(-1, 1, (m, n)).astype(dtype)
    As, Bs = (A if ta == 111 else A.T), (B if tb == 111 else B.T)
    pad = (m + n) % 2
    lda, ldb, ldc = ((x.shape[0] if order == COL else x.shape[1]) + pad for x in (As, Bs, C))
    a, b, c = (store(order, x, ld).astype(dtype) for x, ld in ((As, lda), (Bs, ldb), (C, ldc)))
    f = zh.cblas_dgemm if dtype == np.float64 else zh.cblas_sgemm
    f(order, ta, tb, m, n, k, alpha, P(a), lda, P(b), ldb, beta, P(c), ldc)
    wide = np.longdouble if dtype == np.float64 else np.float64
    ref = alpha * (A.astype(wide) @ B.astype(wide)) + beta * C.astype(wide)
    u = np.finfo(dtype).eps / 2
    bound = (k + 4) * u * (abs(alpha) * (np.abs(A).astype(wide) @ np.abs(B).astype(wide)) + abs(beta) * np.abs(C))
    assert np.all(np.abs(dense(order, m, n, c.astype(np.float64), ldc) - ref) <= bound + np.finfo(dtype).tiny)


@pytest.mark.parametrize("uplo", [121, 122])
@pytest.mark.parametrize("n,k", [(64, 1000), (65, 2000), (200, 600)])
def test_syrk_split(zh, uplo, n, k):
    rng = np.random.default_rng(n + k)
    A, C = rng.uniform(-1, 1, (n, k)), rng.uniform(-1, 1, (n, n))
    a, c = store(COL, A, n), store(COL, C, n)
    zh.cblas_dsyrk(COL, uplo, 111, n, k, -1.0, P(a), n, 1.0, P(c), n)
    got = dense(COL, n, n, c, n)
    L = A.astype(np.longdouble)
    ref, bound = C - L @ L.T, (k + 4) * 2.0 ** -53 * (np.abs(L) @ np.abs(L).T + np.abs(C))
    tri = np.tril(np.ones((n, n), bool)) if uplo == 122 else np.triu(np.ones((n, n), bool))
    assert np.all(np.abs(got - ref)[tri] <= bound[tri])
    assert np.array_equal(got[~tri], C[~tri])


def test_many_workgroup_rounds_match_between_tiles(zh, torch_cuda):
    """Around the line between the tile sizes both kernels give the same bits (the
    load-unit kernel switched off and on)."""
    torch = torch_cuda
    import ctypes
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for m, n, k in ((1920, 1920, 64), (2048, 2176, 48), (2048, 2048, 32), (2500, 2500, 32)):
        g = torch.Generator(device="cuda")
        g.manual_seed(m + n)
        a, b = (torch.rand(x, dtype=torch.float64, device="cuda", generator=g) - 0.5 for x in ((k, m), (n, k)))
        out = []
        for on in (0, 1):
            c = torch.ones(n, m, dtype=torch.float64, device="cuda")
            was = zh.zmlhip_set_gemm_lds_dma(on)
            try:
                assert zh.zmlhip_dgemm(COL, 111, 111, m, n, k, -1.0, P(a), m, P(b), k, 1.0, P(c), m, s) == 0
            finally:
                zh.zmlhip_set_gemm_lds_dma(was)
            out.append(c)
        torch.cuda.synchronize()
        assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("transa,transb", [(111, 111), (112, 111), (111, 112), (112, 112)])
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (-1.0, 1.0), (0.5, 2.0)])
def test_fp32_load_unit_kernel(zh, torch_cuda, transa, transb, alpha, beta):
    """FP32 products on the load unit: ragged tiles in both directions (the last
    four rows or columns alone in theirs), one slab and several. The same bits as
    with the load-unit kernel off, and within k u of the sum of the products'
    magnitudes (u = 2^-24, gamma_k) of the FP64 product."""
    torch = torch_cuda
    import ctypes
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for m, n, k in ((2048, 2048, 32), (2436, 2564, 96), (4100, 2052, 160)):
        g = torch.Generator(device="cuda")
        g.manual_seed(m + k)
        sa = (k, m) if transa == 111 else (m, k)     # column-major storage seen as rows
        sb = (n, k) if transb == 111 else (k, n)
        a, b, c0 = (torch.rand(x, dtype=torch.float32, device="cuda", generator=g) - 0.5 for x in (sa, sb, (n, m)))
        out = []
        for on in (0, 1):
            c = c0.clone()
            was = zh.zmlhip_set_gemm_lds_dma(on)
            try:
                assert zh.zmlhip_sgemm(COL, transa, transb, m, n, k, alpha, P(a), sa[1], P(b), sb[1], beta, P(c), m, s) == 0
            finally:
                zh.zmlhip_set_gemm_lds_dma(was)
            out.append(c)
        torch.cuda.synchronize()
        assert torch.equal(out[0], out[1])
        A = (a.t() if transa == 111 else a).double()     # m x k
        Bm = (b.t() if transb == 111 else b).double()    # k x n
        ref = alpha * (A @ Bm) + beta * c0.t().double()
        mag = abs(alpha) * (A.abs() @ Bm.abs()) + abs(beta) * c0.t().double().abs()
        assert bool(((out[1].t().double() - ref).abs() <= (k + 3) * 2.0 ** -24 * mag).all())
