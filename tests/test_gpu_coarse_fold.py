"""Plain products whose K the tile classes would split in coarse pieces keep that
split's sums where the kernel that divides K among wavefronts takes them: blocks
of 128 k in order within a piece, then the pieces in order, bit for bit.  One k of
each block holds a number, the others zero, so that a block's sum is that number
and NumPy's FP32 adds give the fold."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(138, 4361, 1479), (417, 4383, 647), (305, 2363, 1713), (1280, 3315, 1016),
          (130, 3886, 4964), (398, 3886, 4199), (1362, 1593, 1418), (85, 5908, 2942)]


def _pieces(ompblas, m, n, k):
    """k per piece, from the partial sums that a request reserves."""
    r = ompblas.Request(ompblas.REQ_GEMM, ompblas.PLAIN_F32, m, n, k, 0.0, 256, 256, 256, 0)
    pieces = ompblas.serve_request_bytes(r) // (4 * m * n)
    chunk = -(-(-(-k // pieces)) // 128) * 128
    assert pieces > 1 and chunk > 128 and -(-k // chunk) == pieces
    return chunk


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_pieces_are_summed_apart(dev, ompblas, m, n, k):
    chunk = _pieces(ompblas, m, n, k)
    rng = np.random.default_rng(k)
    blocks = -(-k // 128)
    v = (rng.uniform(-1, 1, (m, blocks)) * 10.0 ** rng.integers(-3, 4, (m, blocks)))
    v = v.astype(np.float32)
    at = np.minimum(128 * np.arange(blocks) + rng.integers(0, 128, blocks), k - 1)
    want = None
    for p in range(0, blocks, chunk // 128):
        piece = np.zeros(m, np.float32)
        for b in range(p, min(blocks, p + chunk // 128)):
            piece = piece + v[:, b]
        want = piece if want is None else want + piece
    assert want.dtype == np.float32
    a = torch.zeros(m, k, device=dev)
    a[:, torch.from_numpy(at).to(dev)] = torch.from_numpy(v).to(dev)
    b = torch.ones(k, n, device=dev)
    at_, bt = a.t().contiguous(), b.t().contiguous()
    w = torch.from_numpy(want).to(dev)[:, None].expand(m, n)
    for pa, ra, ca in ((a, k, 1), (at_, 1, m)):
        for pb, rb, cb in ((b, n, 1), (bt, 1, k)):
            c = torch.full((m, n), float("nan"), device=dev)
            ompblas.check(ompblas.sgemm(m, n, k, 1.0, pa.data_ptr(), ra, ca, pb.data_ptr(), rb, cb,
                                        0.0, c.data_ptr(), n, 1, 0))
            assert torch.equal(c, w)
