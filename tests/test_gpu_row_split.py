"""The row splits of the rank-1 update and of the line copy (a transpose
between storage orders): row lengths around the lines between them, rows
that start anywhere in a 128-byte line, and updates on both sides of the
streaming limit.  Every element is one fma or a copy, so the results are
exact: integers for the update, bits for the copy."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [
    (5, 1), (3, 31), (7, 33), (1100, 511), (9, 512), (1027, 513), (5, 1023), (1030, 1024),
    (6, 1025), (3, 1059), (4, 4099), (2000, 4096 * 3 + 37)])
@pytest.mark.parametrize("order", ["C", "F"])
@pytest.mark.parametrize("off", [0, 5])
def test_rows_of_every_split(dev, ompblas, rows, cols, order, off):
    def view(values):  # a rows x cols view of leading dimension cols + off, inside a guarded buffer
        buf = torch.full((rows * (cols + off) + off,), -7.0, device=dev)
        v = buf[off:].view(rows, cols + off)[:, :cols]
        v.copy_(values)
        return buf, v

    g = torch.Generator(device=dev).manual_seed(3)
    x = torch.randint(-50, 50, (rows,), device=dev, generator=g).float()
    y = torch.randint(-50, 50, (cols,), device=dev, generator=g).float()
    c0 = torch.randint(-50, 50, (rows, cols), device=dev, generator=g).float()
    buf, c = view(c0)
    guard = buf.clone()
    if order == "C":
        ompblas.outer_prod(c, x, y)()
    else:
        ompblas.outer_prod(c.t(), y, x)()
    guard[off:].view(rows, cols + off)[:, :cols] = c0 + x[:, None] * y[None, :]
    assert torch.equal(buf, guard)

    # A column-major into C row-major (and the other way round): a line copy
    src_buf, src = view(c0)
    dst_buf, dst = view(torch.zeros_like(c0))
    guard = dst_buf.clone()
    if order == "C":
        ompblas.transpose(dst, src.t())()
    else:
        ompblas.transpose(dst.t(), src)()
    guard[off:].view(rows, cols + off)[:, :cols] = c0
    assert torch.equal(dst_buf, guard)
