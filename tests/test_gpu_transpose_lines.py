"""Out-of-place transpose through whole-line tiles: extents around the edges
of both tile shapes, rows of C that start anywhere in a 128-byte line, leading
dimensions on and off lines, and rows 32 KB apart (the diagonal tile order).
A transpose moves bits, so every comparison is exact, the guard around C
included."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,pad,off", [
    (1, 1, 0, 0), (1, 70, 0, 3), (70, 1, 2, 0), (31, 33, 0, 1), (32, 32, 0, 0), (33, 31, 1, 31),
    (64, 32, 0, 0), (65, 33, 7, 5), (63, 65, 1, 30), (96, 64, 32, 32), (95, 127, 33, 2),
    (300, 3, 0, 17), (3, 300, 0, 17), (257, 129, 63, 0),
    (4096, 4096, 0, 0), (4097, 4099, 0, 0), (4127, 4100, 5, 9), (131, 128200, 0, 1),
    (128200, 131, 0, 1), (8192, 2049, 0, 0), (8192, 2048, 0, 7)])
@pytest.mark.parametrize("order", ["C", "F"])
def test_transpose_any_line_offset(dev, ompblas, m, n, pad, off, order):
    src = torch.arange(m * (n + pad), device=dev, dtype=torch.int32).view(torch.float32)
    a = src.view(m, n + pad)[:, :n]
    buf = torch.full((n * (m + pad) + off,), -1, device=dev, dtype=torch.int32)
    guard = buf.clone()
    c = buf.view(torch.float32)[off:].view(n, m + pad)[:, :m]
    if order == "C":
        ompblas.transpose(c, a)()
    else:
        ompblas.transpose(c.t(), a.t())()
    guard[off:].view(n, m + pad)[:, :m] = \
        src.view(torch.int32).view(m, n + pad)[:, :n].t()
    assert torch.equal(buf, guard)
