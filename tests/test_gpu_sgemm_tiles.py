"""Plain SGEMM at the edges of its tiles and slices, in every layout of A and B,
at any alignment: its loads are clamped into the operands rather than guarded.
Integer operands make every sum exact; what lies around the operands is NaN."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def operand(dev, g, rows, cols, row_major, pad, off):
    """An integer rows x cols view, `off` floats into a buffer of NaN with `pad`
    floats between its lines."""
    lines, width = (rows, cols) if row_major else (cols, rows)
    buf = torch.full((off + (lines - 1) * (width + pad) + width + 64,), float("nan"), device=dev)
    v = torch.as_strided(buf, (lines, width), (width + pad, 1), off)
    v.copy_(torch.randint(-8, 9, (lines, width), device=dev, generator=g))
    return v if row_major else v.t()


def product(ompblas, a, b, alpha=1.0, beta=0.0, c0=None):
    (m, k), n = a.shape, b.shape[1]
    c = torch.full((m, n), float("nan"), device=a.device) if c0 is None else c0.clone()
    ompblas.check(ompblas.sgemm(m, n, k, alpha, a.data_ptr(), a.stride(0), a.stride(1),
                                b.data_ptr(), b.stride(0), b.stride(1), beta, c.data_ptr(), n, 1,
                                0))
    return c


@pytest.mark.parametrize("a_row", [True, False])
@pytest.mark.parametrize("b_row", [True, False])
@pytest.mark.parametrize("k", [1, 2, 3, 15, 16, 17, 31, 33, 127, 128, 129, 144, 513])
@pytest.mark.parametrize("pad,off", [(0, 0), (0, 1), (1, 2), (4, 0)])
def test_edges(dev, ompblas, a_row, b_row, k, pad, off):
    g = torch.Generator(device=dev).manual_seed(k * 16 + pad)
    for m, n in ((1, 1), (1, 5), (2, 3), (3, 2), (3, 65), (4, 63), (63, 4), (65, 1), (64, 64),
                 (67, 129), (127, 61), (128, 128), (130, 257), (1027, 1409), (2305, 3074)):
        if m > 2000 and k not in (16, 33, 129):  # the largest tile class
            continue
        a = operand(dev, g, m, k, a_row, pad, off)
        b = operand(dev, g, k, n, b_row, pad, off)
        want = a.double() @ b.double()
        assert torch.equal(product(ompblas, a, b).double(), want), (m, n)
        c0 = torch.randint(-8, 9, (m, n), device=dev, generator=g).float()
        got = product(ompblas, a, b, -2.0, 3.0, c0)
        assert torch.equal(got.double(), -2 * want + 3 * c0), (m, n)


@pytest.mark.parametrize("ld", [(1 << 23) - 2, (1 << 23) + 3])
def test_lines_far_apart(dev, ompblas, ld):
    """Tiles whose lines span less and more than 32-bit byte offsets reach."""
    m, n, k = 130, 129, 150
    g = torch.Generator(device=dev).manual_seed(5)
    buf = torch.empty(m * ld, device=dev)
    far = torch.as_strided(buf, (m, k), (ld, 1))
    far.copy_(torch.randint(-8, 9, (m, k), device=dev, generator=g))
    near = torch.randint(-8, 9, (k, n), device=dev, generator=g).float()
    want = far.double() @ near.double()
    assert torch.equal(product(ompblas, far, near).double(), want)
    assert torch.equal(product(ompblas, near.t(), far.t()).double(), want.t())


@pytest.mark.parametrize("a_row", [True, False])
@pytest.mark.parametrize("b_row", [True, False])
def test_k_divided_among_wavefronts(dev, ompblas, a_row, b_row):
    """Sizes where a workgroup's wavefronts share K, in 32 x 32 and 64 x 64
    tiles: rounds of 2, 4 and 8 blocks of 128, the last one partial or short."""
    g = torch.Generator(device=dev).manual_seed(23)
    for m, n in ((32, 32), (33, 31), (1, 70), (200, 150), (515, 513), (1024, 1022), (961, 963)):
        for k in (5, 112, 128, 130, 256, 257, 500, 1024, 1025, 1160, 2175):
            a = operand(dev, g, m, k, a_row, 1, 1)
            b = operand(dev, g, k, n, b_row, 0, 3)
            want = a.double() @ b.double()
            assert torch.equal(product(ompblas, a, b).double(), want), (m, n, k)
            c0 = torch.randint(-8, 9, (m, n), device=dev, generator=g).float()
            got = product(ompblas, a, b, 0.5, -1.0, c0)
            assert torch.equal(got.double(), want / 2 - c0), (m, n, k)


@pytest.mark.parametrize("m,n,k", [(31, 33, 129), (150, 200, 301), (512, 512, 512), (515, 300, 900),
                                   (1024, 1024, 1024), (960, 1000, 1900)])
def test_bits_of_the_unsplit_sum(dev, ompblas, m, n, k):
    """The wavefronts' block sums meet in block order: the bits of a grouped
    launch, whose tiles run through all of K."""
    g = torch.Generator(device=dev).manual_seed(k)
    a = torch.rand((m, k), device=dev, generator=g) * 2 - 1
    b = torch.rand((k, n), device=dev, generator=g) * 2 - 1
    c0 = torch.rand((m, n), device=dev, generator=g)
    for alpha, beta in ((1.0, 0.0), (1.5, -0.5)):
        c = c0.clone()
        plan = ompblas.GroupPlan([(m, n, k, a.data_ptr(), k, b.data_ptr(), n, c.data_ptr(), n,
                                   alpha, beta)], [])
        plan.launch()
        torch.cuda.synchronize()
        assert torch.equal(product(ompblas, a, b, alpha, beta, c0), c)
