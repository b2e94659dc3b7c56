"""Plain products whose k steps lie less than 4 floats apart (one to three
columns of B, contiguous): the slices that unguarded loads must leave at the end
of K may lie in the accumulation block before the last.  Integer operands, exact."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [127, 129, 130, 131, 257, 258, 386, 1025])
@pytest.mark.parametrize("m,n", [(100, 1), (1, 100), (70, 2), (65, 3), (2, 65), (4100, 1)])
def test_few_lines(dev, ompblas, m, n, k):
    g = torch.Generator(device=dev).manual_seed(k)
    a = torch.randint(-8, 9, (m, k), device=dev, generator=g).float()
    b = torch.randint(-8, 9, (k, n), device=dev, generator=g).float()
    want = a.double() @ b.double()
    at, bt = a.t().contiguous(), b.t().contiguous()   # column-major forms
    for (pa, ra, ca) in ((a, k, 1), (at, 1, m)):
        for (pb, rb, cb) in ((b, n, 1), (bt, 1, k)):
            c = torch.full((m, n), float("nan"), device=dev)
            ompblas.check(ompblas.sgemm(m, n, k, 1.0, pa.data_ptr(), ra, ca, pb.data_ptr(), rb, cb,
                                        0.0, c.data_ptr(), n, 1, 0))
            assert torch.equal(c.double(), want)
    c = torch.full((m, n), float("nan"), device=dev)
    plan = ompblas.GroupPlan([(m, n, k, a.data_ptr(), k, b.data_ptr(), n, c.data_ptr(), n, 1.0,
                               0.0)], [])
    plan.launch()
    torch.cuda.synchronize()
    assert torch.equal(c.double(), want)
