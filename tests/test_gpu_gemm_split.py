"""Products whose k is split over workgroups (few tiles, long k) as a caller of an
asynchronous call meets them: the same bits when the call is recorded into a graph
(where nothing may be allocated) as when it is made directly, nothing waited for on
the way, and no effect on a capture that another thread has under way."""
import ctypes
import threading

import pytest

from tests.helpers import COL, P

pytestmark = pytest.mark.gpu

N, T = 111, 112
SHAPES = [(64, 64, 4100), (33, 70, 600), (124, 130, 2000), (1, 130, 1111), (200, 180, 512)]


def stream(torch):
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def operands(torch, m, n, k, dtype, ta=N, tb=N):
    g = torch.Generator(device="cuda")
    g.manual_seed(m + n + k)
    sa, sb = ((k, m) if ta == N else (m, k)), ((n, k) if tb == N else (k, n))   # column-major storage seen as rows
    return [torch.rand(x, dtype=dtype, device="cuda", generator=g).sub_(0.5) for x in (sa, sb, (n, m))]


def product(zh, torch, m, n, k, a, b, c, alpha, beta, ta=N, tb=N):
    f = zh.zmlhip_dgemm if a.dtype == torch.float64 else zh.zmlhip_sgemm
    assert f(COL, ta, tb, m, n, k, alpha, P(a), a.shape[1], P(b), b.shape[1], beta, P(c), m, stream(torch)) == 0


def capture(torch, call, **kw):
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(graph, stream=side, **kw):
        call()
    return graph


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("ta,tb", [(N, N), (T, N), (N, T), (T, T)])
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (-1.0, 1.0), (0.7, 0.3)])
def test_a_recorded_product_has_the_direct_ones_bits(zh, torch_cuda, dtype, ta, tb, alpha, beta):
    torch = torch_cuda
    dtype = getattr(torch, dtype)
    for m, n, k in SHAPES:
        a, b, c0 = operands(torch, m, n, k, dtype, ta, tb)
        want, got = c0.clone(), c0.clone()
        product(zh, torch, m, n, k, a, b, want, alpha, beta, ta, tb)
        torch.cuda.synchronize()
        graph = capture(torch, lambda: product(zh, torch, m, n, k, a, b, got, alpha, beta, ta, tb))
        for _ in range(3):
            got.copy_(c0)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(got, want), (m, n, k)


@pytest.mark.parametrize("uplo", [121, 122])
@pytest.mark.parametrize("n,k", [(65, 2000), (200, 600)])
def test_a_recorded_syrk_has_the_direct_ones_bits(zh, torch_cuda, uplo, n, k):
    torch = torch_cuda
    a, _, _ = operands(torch, n, n, k, torch.float64)
    c0 = torch.rand(n, n, dtype=torch.float64, device="cuda")
    want, got = c0.clone(), c0.clone()

    def call(c):
        assert zh.zmlhip_dsyrk(COL, uplo, N, n, k, 0.7, P(a), n, 0.3, P(c), n, stream(torch)) == 0

    call(want)
    torch.cuda.synchronize()
    graph = capture(torch, lambda: call(got))
    for _ in range(3):
        got.copy_(c0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)


def in_new_thread(work):
    """Runs work on a thread that has no workspaces of the library yet."""
    out, wrong = [], []

    def run():
        try:
            out.append(work())
        except BaseException as e:
            wrong.append(e)

    t = threading.Thread(target=run)
    t.start()
    t.join()
    if wrong:
        raise wrong[0]
    return out[0]


def test_products_of_growing_size_wait_for_nothing(zh, torch_cuda):
    torch = torch_cuda
    sizes = [(64, 64, 1024), (300, 300, 1024), (900, 800, 1024)]
    sets = [operands(torch, m, n, k, torch.float64) for m, n, k in sizes]
    for (m, n, k), (a, b, c) in zip(sizes, sets):
        product(zh, torch, m, n, k, a, b, c, 1.0, 0.0)
    torch.cuda.synchronize()

    def work():
        busy, done = torch.cuda.Stream(), torch.cuda.Event()
        with torch.cuda.stream(busy):
            torch.cuda._sleep(1_000_000_000)   # about half a second of a kernel that only counts
            done.record()
        with torch.cuda.stream(torch.cuda.Stream()):
            for (m, n, k), (a, b, c) in zip(sizes, sets):
                product(zh, torch, m, n, k, a, b, c, 1.0, 0.0)
        return done.query()

    finished = in_new_thread(work)
    torch.cuda.synchronize()
    assert not finished


@pytest.mark.parametrize("ends", ["after", "during"])
def test_a_product_leaves_another_threads_capture_alone(zh, torch_cuda, ends):
    """A first product (which allocates) on a thread that ends after the other thread's
    capture, or during it (which frees)."""
    torch = torch_cuda
    m, n, k = 64, 64, 4096
    a, b, c = operands(torch, m, n, k, torch.float64)
    want = c.clone()
    product(zh, torch, m, n, k, a, b, want, 1.0, 0.0)
    x = torch.ones(1000, device="cuda")
    other = torch.cuda.Stream()
    args = (COL, N, N, m, n, k, 1.0, P(a), m, P(b), k, 0.0, P(c), m, ctypes.c_void_p(other.cuda_stream))
    torch.cuda.synchronize()
    called, captured, rc = threading.Event(), threading.Event(), []

    def work():
        rc.append(zh.zmlhip_dgemm(*args))
        called.set()
        if ends == "after":
            captured.wait(30)

    thread = threading.Thread(target=work)

    def call():
        x.add_(1)
        thread.start()
        called.wait(30)
        if ends == "during":
            thread.join()
        x.add_(1)

    try:
        graph = capture(torch, call, capture_error_mode="global")
    finally:
        captured.set()
        thread.join()
    torch.cuda.synchronize()
    assert rc == [0] and torch.equal(c, want)
    for _ in range(3):
        graph.replay()
    torch.cuda.synchronize()
    assert float(x[0]) == 7.0
