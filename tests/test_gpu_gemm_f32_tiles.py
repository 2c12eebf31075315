"""FP32 products around the line k = 128 between the 64 x 64 tiles and the load
unit's 128 x 128 ones: ragged tiles in both directions, several slabs, the same
bits from both, and the choice no slower than the tiles it leaves out."""
import ctypes

import pytest

from tests.helpers import COL, P

pytestmark = pytest.mark.gpu


def call(zh, torch, m, n, k, transa, transb, alpha, beta, a, b, c):
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert zh.zmlhip_sgemm(COL, transa, transb, m, n, k, alpha, P(a), a.shape[1], P(b), b.shape[1], beta, P(c), m, s) == 0


def operands(torch, m, n, k, transa=111, transb=111):
    g = torch.Generator(device="cuda")
    g.manual_seed(m + k)
    shapes = ((k, m) if transa == 111 else (m, k)), ((n, k) if transb == 111 else (k, n)), (n, m)
    return [torch.rand(x, dtype=torch.float32, device="cuda", generator=g) - 0.5 for x in shapes]


@pytest.mark.parametrize("transa,transb", [(111, 111), (112, 111), (111, 112), (112, 112)])
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (-1.0, 1.0), (0.5, 2.0)])
@pytest.mark.parametrize("m,n,k", [(2436, 2564, 128), (2436, 2564, 160), (3840, 3844, 288)])
def test_both_kernels_give_the_same_bits(zh, torch_cuda, transa, transb, alpha, beta, m, n, k):
    torch = torch_cuda
    a, b, c0 = operands(torch, m, n, k, transa, transb)
    out = []
    for on in (0, 1):
        c = c0.clone()
        was = zh.zmlhip_set_gemm_lds_dma(on)
        try:
            call(zh, torch, m, n, k, transa, transb, alpha, beta, a, b, c)
        finally:
            zh.zmlhip_set_gemm_lds_dma(was)
        out.append(c)
    torch.cuda.synchronize()
    assert torch.equal(out[0], out[1])
    # within (k + 3) u of the sum of the products' magnitudes (gamma_k, the scaling and the sum)
    A, B = (a.t() if transa == 111 else a).double(), (b.t() if transb == 111 else b).double()
    ref = alpha * (A @ B) + beta * c0.t().double()
    mag = abs(alpha) * (A.abs() @ B.abs()) + abs(beta) * c0.t().double().abs()
    assert bool(((out[1].t().double() - ref).abs() <= (k + 3) * 2.0 ** -24 * mag).all())


@pytest.mark.parametrize("k", [64, 128])
def test_a_short_k_takes_the_faster_tiles(zh, torch_cuda, k):
    """6000 x 6000: the larger tiles took 1.2 to 1.4 times as long here."""
    torch = torch_cuda
    m = n = 6000
    a, b, c = operands(torch, m, n, k)
    best = {0: float("inf"), 1: float("inf")}
    for _ in range(15):
        for on in (0, 1):
            was = zh.zmlhip_set_gemm_lds_dma(on)
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            try:
                e0.record()
                call(zh, torch, m, n, k, 111, 111, 1.0, 0.0, a, b, c)
                e1.record()
            finally:
                zh.zmlhip_set_gemm_lds_dma(was)
            torch.cuda.synchronize()
            best[on] = min(best[on], e0.elapsed_time(e1))
    assert best[1] <= 1.1 * best[0]
