"""Thin operands with more tiles than one launch may have work-items for (2^32): the
transpose strides over its tiles."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _room(nbytes):
    free, _ = torch.cuda.mem_get_info()
    if free < nbytes:
        pytest.skip("not enough memory free")


def test_transpose_of_thin_matrix(dev, ompblas):
    rows, cols = 2, 1 << 30
    _room(40 << 30)
    a = torch.empty(rows, cols, device=dev)
    ompblas.fill_uniform(a, 95, 0)
    c = torch.full((cols, rows), float("nan"), device=dev)
    ompblas.check(ompblas.stranspose(rows, cols, a.data_ptr(), cols, 1, c.data_ptr(), rows, 1))
    torch.cuda.synchronize()
    for r in range(rows):
        assert torch.equal(c[:, r], a[r])
