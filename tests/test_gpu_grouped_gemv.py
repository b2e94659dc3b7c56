"""Grouped GEMV items where the number of rows at once and of loads per row changes,
and at the edges of rounds and of a wavefront's rows: exact on integers, the bits of
the direct call on others, and nothing read past a row (the padding is NaN)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

MS = (1, 3, 4, 5, 15, 17, 65, 130)
NS = (1, 3, 4, 255, 256, 257, 259, 260, 263, 511, 515, 516, 519, 767, 768, 769, 773, 1023, 1024, 1027,
      1028, 1283, 1537, 1795, 2048, 2052, 3001, 4095)


@pytest.mark.parametrize("pad,off", [(0, 0), (1, 1), (5, 2)])
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (-2.0, 0.5)])
def test_item_edges(dev, ompblas, pad, off, alpha, beta):
    g = torch.Generator(device=dev).manual_seed(pad)
    for real in (False, True):
        def values(*shape):
            return (torch.rand(shape, device=dev, generator=g) * 2 - 1 if real else
                    torch.randint(-8, 9, shape, device=dev, generator=g).float())

        ops = []
        for m in MS:
            for n in NS:
                a = torch.as_strided(torch.full((off + m * (n + pad) + 64,), float("nan"), device=dev),
                                     (m, n), (n + pad, 1), off)
                ops.append((a.copy_(values(m, n)), values(n), values(m)))
        wants = [alpha * (a.double() @ x.double()) + beta * y.double() for a, x, y in ops]
        direct = [y.clone() for _, _, y in ops]
        plan = ompblas.GroupPlan([], [(a.shape[0], a.shape[1], a.data_ptr(), a.stride(0), x.data_ptr(),
                                       y.data_ptr(), alpha, beta) for a, x, y in ops], 0)
        plan.launch()
        for (a, x, y), d, want in zip(ops, direct, wants):
            m, n = a.shape
            ompblas.check(ompblas.sgemv(m, n, alpha, a.data_ptr(), a.stride(0), 1, x.data_ptr(), beta,
                                        d.data_ptr()))
            torch.cuda.synchronize()
            assert torch.equal(y, d), (m, n)
            if not real:
                assert torch.equal(y.double(), want), (m, n)
