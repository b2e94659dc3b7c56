"""Column-major GEMV around the edges of its row blocks (4, 64 and 256 rows),
column rounds and chunks.  Integer operands keep every sum below 2^24, so the
results are exact in any order of adds; the fallback without arrival counters
gives the same bits on real data."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def view(dev, m, n, off, gen):
    buf = torch.randint(-9, 10, (n * (m + off) + off,), device=dev, generator=gen).float()
    return buf[off:].view(n, m + off)[:, :m].t()


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 63, 64, 65, 257, 1021, 1024, 1025, 1027, 2305])
@pytest.mark.parametrize("n,off", [(1, 0), (2, 3), (63, 1), (64, 0), (127, 5), (129, 0), (1025, 1),
                                   (4111, 0)])
def test_edges_integer_exact(dev, ompblas, m, n, off):
    g = torch.Generator(device=dev).manual_seed(m * 8191 + n)
    a = view(dev, m, n, off, g)
    x = torch.randint(-9, 10, (n,), device=dev, generator=g).float()
    y0 = torch.randint(-9, 10, (m,), device=dev, generator=g).float()
    for alpha, beta in ((1.0, 1.0), (-2.0, 0.0), (2.0, -3.0)):
        y = y0.clone() if beta else torch.full_like(y0, float("nan"))
        ompblas.check(ompblas.sgemv(m, n, alpha, a.data_ptr(), 1, m + off, x.data_ptr(), beta,
                                    y.data_ptr()))
        want = alpha * (a.double() @ x.double()) + (beta * y0.double() if beta else 0)
        assert torch.equal(y.double(), want), (alpha, beta)


def test_streamed_operand_and_special_values(dev, ompblas):
    """Past the streaming limit (120 MB), and an infinity in the last column,
    which clamped loads of the last round repeat: only its own row sees it."""
    m, n = 5001, 6001
    g = torch.Generator(device=dev).manual_seed(5)
    a = view(dev, m, n, 0, g)
    x = torch.randint(-9, 10, (n,), device=dev, generator=g).float()
    x[-1] = 3.0
    want = a.double() @ x.double()
    y = torch.zeros(m, device=dev)
    ompblas.mtv(y, a, x)()
    assert torch.equal(y.double(), want)
    a[7, -1] = float("inf")
    y.zero_()
    ompblas.mtv(y, a, x)()
    want[7] = float("inf")
    assert torch.equal(y.double(), want)


def test_streams_past_the_counters_give_the_same_bits(dev, ompblas):
    lib = ompblas.lib()
    shapes = ((9003, 601), (700, 3001), (3, 5000))
    cases = []
    for i, (m, n) in enumerate(shapes):
        a, x = torch.empty(n, m, device=dev), torch.empty(n, device=dev)
        ompblas.fill_uniform(a, 91, 2 * i)
        ompblas.fill_uniform(x, 91, 2 * i + 1)
        cases.append((m, n, a, x))
    hip = ctypes.CDLL("libamdhip64.so")
    streams = []
    for _ in range(70):
        s = ctypes.c_void_p()
        assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0
        streams.append(s)
    torch.cuda.synchronize()
    outs = []
    for s in streams:
        for m, n, a, x in cases:
            y = torch.empty(m, device=dev)
            torch.cuda.current_stream().synchronize()
            ompblas.check(lib.omb_sgemv(m, n, 1.0, a.data_ptr(), 1, m, x.data_ptr(), 0.0,
                                        y.data_ptr(), s))
            outs.append(y)
    torch.cuda.synchronize()
    for i, y in enumerate(outs):
        assert torch.equal(y, outs[i % len(cases)])
    for s in streams:
        assert hip.hipStreamDestroy(s) == 0
