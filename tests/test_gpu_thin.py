"""Thin operands, whose kernels are chosen by their short side: GEMV of few long
rows or few tall columns, transposes that are one row or one column of tiles.
Integer operands keep sums exact; a transpose moves bits, its surroundings
included."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 3, 17, 512, 513])
@pytest.mark.parametrize("n,off", [(10240, 0), (10241, 1), (12003, 0), (34882, 3)])
def test_few_long_rows(dev, ompblas, m, n, off):
    g = torch.Generator(device=dev).manual_seed(m * 31 + n)
    lda = n + off
    for make in (lambda k: torch.randint(-9, 10, (k,), device=dev, generator=g).float(),
                 lambda k: torch.rand(k, device=dev, generator=g) * 2 - 1):
        buf = make(m * lda + off)
        a, x, y0 = buf[off:].view(m, lda)[:, :n], make(n), make(m)
        y, z = y0.clone(), y0.clone()
        ompblas.check(ompblas.sgemv(m, n, -2.0, a.data_ptr(), lda, 1, x.data_ptr(), 1.5,
                                    y.data_ptr()))
        plan = ompblas.GroupPlan([], [(m, n, a.data_ptr(), lda, x.data_ptr(), z.data_ptr(), -2.0,
                                       1.5)])
        plan.launch()
        torch.cuda.synchronize()
        assert torch.equal(y, z)  # the grouped item's bits
        want = -2.0 * (a.double() @ x.double()) + 1.5 * y0.double()
        err = (y.double() - want).abs().max().item()
        assert err <= 2.0 * n * 2.0 ** -24 * 2.0 * a.abs().double().matmul(x.abs().double()).max().item()
        if buf[0].item() == round(buf[0].item()):
            assert torch.equal(y.double(), want)


@pytest.mark.parametrize("m", [5, 1024, 1025, 65280, 65281, 65537, 163474])
@pytest.mark.parametrize("n,off", [(1, 0), (4, 1), (5, 0), (16, 3), (17, 0), (32, 0), (33, 1),
                                   (64, 0), (65, 0), (128, 1), (129, 0), (256, 3), (257, 0)])
def test_few_columns(dev, ompblas, m, n, off):
    g = torch.Generator(device=dev).manual_seed(m + n)
    ld = m + off
    buf = torch.randint(-9, 10, (n * ld + off,), device=dev, generator=g).float()
    a = buf[off:].view(n, ld)[:, :m].t()
    x = torch.randint(-9, 10, (n,), device=dev, generator=g).float()
    y0 = torch.randint(-9, 10, (m,), device=dev, generator=g).float()
    for alpha, beta in ((1.0, 1.0), (-2.0, 0.0)):
        y = y0.clone() if beta else torch.full_like(y0, float("nan"))
        ompblas.check(ompblas.sgemv(m, n, alpha, a.data_ptr(), 1, ld, x.data_ptr(), beta,
                                    y.data_ptr()))
        want = alpha * (a.double() @ x.double()) + beta * y0.double()
        assert torch.equal(y.double(), want)


@pytest.mark.parametrize("m,n", [(1, 70001), (4, 128000), (9, 70000), (10, 6401), (11, 70001),
                                 (31, 6400), (33, 70016), (40, 70001), (63, 70016), (64, 70001),
                                 (64, 300001), (65, 300000), (12, 1500001)])
@pytest.mark.parametrize("pad,off", [(0, 0), (1, 0), (0, 5), (32, 32)])
def test_thin_transpose(dev, ompblas, m, n, pad, off):
    for rows, cols in ((m, n), (n, m)):
        src = torch.arange(rows * (cols + pad), device=dev, dtype=torch.int32).view(torch.float32)
        a = src.view(rows, cols + pad)[:, :cols]
        buf = torch.full((cols * (rows + pad) + off,), -1, device=dev, dtype=torch.int32)
        guard = buf.clone()
        c = buf.view(torch.float32)[off:].view(cols, rows + pad)[:, :rows]
        ompblas.transpose(c, a)()
        guard[off:].view(cols, rows + pad)[:, :rows] = \
            src.view(torch.int32).view(rows, cols + pad)[:, :cols].t()
        assert torch.equal(buf, guard)
