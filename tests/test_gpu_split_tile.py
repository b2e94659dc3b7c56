"""Split products small enough for one launch of 64 x 64 tiles, around the edges of
tiles, slices and accumulation blocks and with K for each number of groups that share
it, in every storage order: exact on integers, and on others the bits of a grouped
item, which keeps the unsplit fold."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [1, 2, 3])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (3, 5, 15), (64, 64, 16), (63, 65, 17), (65, 127, 255),
                                   (128, 40, 256), (40, 200, 257), (200, 150, 301), (33, 500, 513),
                                   (48, 2600, 770), (130, 70, 1024), (2500, 311, 1270)])
def test_split_tiles(dev, ompblas, mode, m, n, k):
    g = torch.Generator(device=dev).manual_seed(m + n + k)

    def matrix(rows, cols, row_major, real):
        shape = (rows, cols + 3) if row_major else (cols, rows + 3)
        v = (torch.rand(shape, device=dev, generator=g) * 2 - 1 if real else
             torch.randint(-4, 5, shape, device=dev, generator=g).float())
        return v[:, :cols] if row_major else v[:, :rows].t()

    for a_row in (True, False):
        for b_row in (True, False):
            for real in (False, True):
                a, b = matrix(m, k, a_row, real), matrix(k, n, b_row, real)
                c = matrix(m, n, True, real)
                got, want = c.clone(), 2.0 * (a.double() @ b.double()) - c.double()
                ompblas.check(ompblas.sgemm(m, n, k, 2.0, a.data_ptr(), a.stride(0), a.stride(1),
                                            b.data_ptr(), b.stride(0), b.stride(1), -1.0,
                                            got.data_ptr(), got.stride(0), 1, mode))
                torch.cuda.synchronize()
                if not real:
                    assert torch.equal(got.double(), want), (a_row, b_row)
                    continue
                ar, br, item = a.contiguous(), b.contiguous(), c.clone()
                ompblas.GroupPlan([(m, n, k, ar.data_ptr(), k, br.data_ptr(), n, item.data_ptr(),
                                    item.stride(0), 2.0, -1.0)], [], mode).launch()
                torch.cuda.synchronize()
                assert torch.equal(got, item), (a_row, b_row)
