"""Thin operands with more tiles or groups of rows than one launch may have
work-items for (2^32): the transpose strides over its tiles, the row maxima of the
scaled split-FP16 product take more than one launch."""
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


@pytest.mark.parametrize("row_major", [False, True])
def test_scaled_fp16_of_many_rows(dev, ompblas, row_major):
    m, n, k = (1 << 27) + 33, 1, 2
    _room(40 << 30)
    g = torch.Generator(device=dev).manual_seed(7)
    lines, width = (m, k) if row_major else (k, m)
    a = torch.randint(-8, 9, (lines, width), device=dev, generator=g, dtype=torch.int8).float()
    b = torch.tensor([[3.0], [-5.0]], device=dev)
    c = torch.full((m, n), float("nan"), device=dev)
    rs, cs = (k, 1) if row_major else (1, m)
    ompblas.check(ompblas.sgemm(m, n, k, 1.0, a.data_ptr(), rs, cs, b.data_ptr(), n, 1, 0.0,
                                c.data_ptr(), n, 1, ompblas.SPLIT_FP16))
    torch.cuda.synchronize()
    cols = (a[:, 0], a[:, 1]) if row_major else (a[0], a[1])
    assert torch.equal(c[:, 0], 3.0 * cols[0] - 5.0 * cols[1])
    del a, c
    torch.cuda.empty_cache()
