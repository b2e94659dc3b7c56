"""Scaled split-FP16 products whose lines differ by large powers of two: a line
maximum that misses an element overflows its FP16 pieces, one that is too
large loses them.  Integers scaled by line keep every sum exact."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("a_row", [True, False])
@pytest.mark.parametrize("b_row", [True, False])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (2, 3, 3), (3, 33, 4), (5, 31, 7), (32, 4, 255),
                                   (33, 65, 257), (130, 36, 1030), (300, 260, 515), (7, 3, 9001),
                                   (64, 35, 33000)])
def test_line_maxima(dev, ompblas, a_row, b_row, m, n, k):
    g = torch.Generator(device=dev).manual_seed(m * 1000 + k)

    def matrix(rows, cols, row_major, scale):
        v = torch.randint(-3, 4, (rows, cols), device=dev, generator=g).float()
        # one large element per line, at its first, last and other places
        for i in range(v.shape[0] if scale.shape[1] == 1 else v.shape[1]):
            at = (i * 37 + (0, -1)[i % 2]) % k
            v[(i, at) if scale.shape[1] == 1 else (at, i)] = 60
        v = v * scale
        return v if row_major else v.t().contiguous().t()

    def powers(shape):
        e = torch.randint(-40, 41, shape, device=dev, generator=g)
        return ((e + 127) << 23).int().view(torch.float32)  # 2^e, exactly

    a = matrix(m, k, a_row, powers((m, 1)))
    b = matrix(k, n, b_row, powers((1, n)))
    c = torch.full((m, n), float("nan"), device=dev)
    ompblas.check(ompblas.sgemm(m, n, k, 1.0, a.data_ptr(), a.stride(0), a.stride(1), b.data_ptr(),
                                b.stride(0), b.stride(1), 0.0, c.data_ptr(), n, 1, 3))
    assert torch.equal(c.double(), a.double() @ b.double())
