"""Writing a split product's tiles back: blocks that end at C's last row or column or
one element to either side of it, alone and in products of several tiles, with and
without a read of C, into a C of a larger leading dimension.  Small integers, so that
every sum is exact in every mode; the padding keeps its value."""
import pytest
import torch

pytestmark = pytest.mark.gpu

MODES = [1, 2, 3]  # split BF16 (6 and 3 products), scaled FP16


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (1.0, 1.0), (2.0, -3.0)])
@pytest.mark.parametrize("m,n,k,pad", [(1, 1, 1, 0), (31, 33, 16, 3), (32, 64, 17, 0),
                                       (63, 65, 40, 1), (64, 64, 16, 0), (65, 63, 40, 5),
                                       (127, 129, 48, 0), (128, 128, 32, 4), (129, 95, 260, 1),
                                       (160, 256, 700, 0), (300, 257, 1030, 7)])
def test_epilogue_edges(dev, ompblas, mode, alpha, beta, m, n, k, pad):
    g = torch.Generator(device=dev).manual_seed(m * 1000 + n)

    def ints(*shape):
        return torch.randint(-4, 5, shape, device=dev, generator=g).float()

    a, b, c = ints(m, k), ints(k, n), ints(m, n + pad)
    want = beta * c.double()[:, :n] + alpha * (a.double() @ b.double())
    if beta == 0.0:
        c[:, :n] = float("nan")  # not read
    got = c.clone()
    ompblas.check(ompblas.sgemm(m, n, k, alpha, a.data_ptr(), k, 1, b.data_ptr(), n, 1, beta,
                                got.data_ptr(), n + pad, 1, mode))
    torch.cuda.synchronize()
    assert torch.equal(got[:, :n].double(), want)
    assert torch.equal(got[:, n:], c[:, n:])
