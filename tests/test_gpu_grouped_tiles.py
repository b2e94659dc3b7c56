"""Grouped GEMM items at the edges of their tiles, slices and accumulation
blocks: exact on integers, and the bits of the direct call in every mode."""
import pytest
import torch

pytestmark = pytest.mark.gpu

MN = ((1, 1), (2, 5), (3, 200), (31, 33), (32, 64), (33, 31), (64, 65), (47, 300), (129, 95))
KS = (1, 3, 15, 16, 17, 33, 127, 128, 130, 255, 257, 300, 385, 512)


@pytest.mark.parametrize("mode", [0, 1, 2, 3])
@pytest.mark.parametrize("pad,off", [(0, 0), (1, 1), (3, 2)])
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (-2.0, 0.5)])
def test_item_edges(dev, ompblas, mode, pad, off, alpha, beta):
    for real in (False, True):
        g = torch.Generator(device=dev).manual_seed(mode * 8 + pad)

        def matrix(rows, cols):
            v = torch.as_strided(torch.full((off + rows * (cols + pad) + 64,), float("nan"), device=dev),
                                 (rows, cols), (cols + pad, 1), off)
            x = (torch.rand((rows, cols), device=dev, generator=g) * 2 - 1 if real else
                 torch.randint(-8, 9, (rows, cols), device=dev, generator=g).float())
            return v.copy_(x)

        ops = [(matrix(m, k), matrix(k, n), matrix(m, n)) for m, n in MN for k in KS]
        direct = [c.clone() for _, _, c in ops]
        gemms = [(a.shape[0], b.shape[1], a.shape[1], a.data_ptr(), a.stride(0), b.data_ptr(),
                  b.stride(0), c.data_ptr(), c.stride(0), alpha, beta) for a, b, c in ops]
        wants = [alpha * (a.double() @ b.double()) + beta * c.double() for a, b, c in ops]
        plan = ompblas.GroupPlan(gemms, [], mode)
        plan.launch()
        for (a, b, c), d, want in zip(ops, direct, wants):
            (m, k), n = a.shape, b.shape[1]
            ompblas.check(ompblas.sgemm(m, n, k, alpha, a.data_ptr(), a.stride(0), 1, b.data_ptr(),
                                        b.stride(0), 1, beta, d.data_ptr(), d.stride(0), 1, mode))
            torch.cuda.synchronize()
            assert torch.equal(c, d), (m, n, k)
            if not real:
                assert torch.equal(c.double(), want), (m, n, k)


@pytest.mark.parametrize("mode", [1, 2, 3])
def test_special_values(dev, ompblas, mode):
    """Infinities, NaN and values past BF16's largest finite one, as in the
    direct call: the same elements are not finite, the others the same bits."""
    g = torch.Generator(device=dev).manual_seed(3)
    for i, v in enumerate((float("inf"), float("-inf"), float("nan"), 3.4e38, -3.3961775e38, 1e-40)):
        m, n, k = 70, 66, 300
        a = torch.rand((m, k), device=dev, generator=g) - 0.5
        b = torch.rand((k, n), device=dev, generator=g) * 1e-3
        a[11 * i % m, 290 if i % 2 else 7] = v
        c, d = torch.zeros((m, n), device=dev), torch.zeros((m, n), device=dev)
        plan = ompblas.GroupPlan([(m, n, k, a.data_ptr(), k, b.data_ptr(), n, c.data_ptr(), n, 1.0,
                                   0.0)], [], mode)
        plan.launch()
        ompblas.check(ompblas.sgemm(m, n, k, 1.0, a.data_ptr(), k, 1, b.data_ptr(), n, 1, 0.0,
                                    d.data_ptr(), n, 1, mode))
        torch.cuda.synchronize()
        assert torch.equal(c.isnan(), d.isnan()) and torch.equal(c.nan_to_num(), d.nan_to_num()), v
        assert torch.isfinite(c).all() == (i > 2), v
