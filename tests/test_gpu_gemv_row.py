"""Row-major GEMV over every row / load split of the launcher: integer operands
keep the sums exact, and on real data the bits are those of the grouped item
(16 rows per wavefront), whose per-row order of adds every split keeps."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 3, 4, 17, 1025, 6143, 6144, 6147, 16384])
@pytest.mark.parametrize("n,off", [(1, 0), (3, 1), (4, 0), (255, 0), (257, 2), (511, 1), (512, 0),
                                   (513, 0), (1024, 0), (1025, 7), (2047, 0), (2049, 1),
                                   (4099, 3)])
def test_every_split_exact_and_grouped_bits(dev, ompblas, m, n, off):
    g = torch.Generator(device=dev).manual_seed(m * 4099 + n)
    lda = n + off

    def check(make):
        buf = make(m * lda + off)
        a, x, y0 = buf[off:].view(m, lda)[:, :n], make(n), make(m)
        outs = []
        for alpha, beta in ((1.0, 0.0), (-2.0, 1.5)):
            y = y0.clone() if beta else torch.full_like(y0, float("nan"))
            ompblas.check(ompblas.sgemv(m, n, alpha, a.data_ptr(), lda, 1, x.data_ptr(), beta,
                                        y.data_ptr()))
            outs.append((alpha, beta, y))
            z = y0.clone()
            plan = ompblas.GroupPlan([], [(m, n, a.data_ptr(), lda, x.data_ptr(), z.data_ptr(),
                                           alpha, beta)])
            plan.launch()
            torch.cuda.synchronize()
            assert torch.equal(y, z)
        return a, x, y0, outs

    a, x, y0, outs = check(lambda k: torch.randint(-9, 10, (k,), device=dev, generator=g).float() * 2)
    for alpha, beta, y in outs:
        want = alpha * (a.double() @ x.double()) + (beta * y0.double() if beta else 0)
        assert torch.equal(y.double(), want)
    check(lambda k: torch.rand(k, device=dev, generator=g) * 2 - 1)


def test_streamed_rows_and_special_values(dev, ompblas):
    """Past the streaming limit, with an infinity in the last whole group of a
    row, which the clamped loads of the last round repeat."""
    for m, n in ((3001, 9001), (9001, 3001)):
        g = torch.Generator(device=dev).manual_seed(7)
        a = torch.randint(-9, 10, (m, n), device=dev, generator=g).float()
        x = torch.randint(1, 10, (n,), device=dev, generator=g).float()
        want = a.double() @ x.double()
        y = torch.zeros(m, device=dev)
        ompblas.mtv(y, a, x)()
        assert torch.equal(y.double(), want)
        a[11, n // 4 * 4 - 1] = float("inf")
        want[11] = float("inf")
        ompblas.mtv(y, a, x)()
        assert torch.equal(y.double(), want)
