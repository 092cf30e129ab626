"""The SpMM's work items and column tiles at their edges (GPU).

Rows of every length around the item and block sizes (1 to 66 values, whole
chunks, chunks with a remainder, a hub row of more than 16 chunks), rows without
values before the first row, in runs of 8 and 9, after a cut row and at the end,
and column counts that take every tile width, among them FP8 rows of an odd number
of 64-column groups.  Every entry is kept (one per 4-column segment, V = 1), so
the reference is the plain product in FP64; an output of L terms in FP32 may be off by
(L + 3) 2^-24 times the sum of the terms' magnitudes (one rounding per FMA, one for
the weight's scale, and the chunk sums).
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import vnm  # noqa: E402

pytestmark = pytest.mark.gpu

HUB = 64 * 17 + 3


@pytest.fixture(scope="module")
def matrix():
    rng = np.random.default_rng(41)
    lens = [0, 0, 0] + list(range(1, 67)) + [0] * 8 + [127] + [0] * 2 + [128, 129] + [1] + [0] * 9 + [HUB, 3] + [0] * 8
    lens += [5] * 40 + [0] * 7
    rows = (len(lens) + 3) // 4 * 4
    segs = HUB + 5
    r, c = [], []
    for i, n in enumerate(lens):
        seg = np.sort(rng.choice(segs, n, replace=False))
        r += [i] * n
        c += list(seg * 4 + rng.integers(0, 4, n))
    R = max(rows, segs * 4)
    v = rng.normal(size=len(r)).astype(np.float32)
    m = vnm.coo_from_tuples(R, R, np.array(r, np.int32), np.array(c, np.int32), v, 4)
    ctx = vnm.Context(0)
    g = vnm.Graph(ctx, m, 4)
    p = g.pack(1, vnm.DT_F32)
    assert p.info().retained_nnz == len(r)
    return m, g, p


def _reference(m, B):
    """(product, sum of magnitudes, terms per row) in FP64."""
    A = torch.sparse_coo_tensor(np.stack([m.row, m.col]), m.val.astype(np.float64), (m.nrows, m.ncols)).to_sparse_csr()
    mag = torch.sparse_coo_tensor(np.stack([m.row, m.col]), np.abs(m.val).astype(np.float64),
                                  (m.nrows, m.ncols)).to_sparse_csr()
    return (A @ B).numpy(), (mag @ B.abs()).numpy(), np.bincount(m.row, minlength=m.nrows)


@pytest.mark.parametrize("dt", [vnm.DT_F32, vnm.DT_BF16, vnm.DT_FP8])
@pytest.mark.parametrize("n", [64, 128, 192, 320, 512])
def test_items_and_tiles_at_their_edges(matrix, dt, n):
    m, g, p = matrix
    gen = torch.Generator().manual_seed(n)
    B = torch.randn(m.ncols, n, generator=gen)
    scales = None
    if dt == vnm.DT_BF16:
        dev = B.to(torch.bfloat16)
        B = dev.double()
    elif dt == vnm.DT_FP8:
        dev = B.to(torch.float8_e4m3fn)
        scales = torch.rand((m.ncols + 127) // 128, generator=gen) + 0.5
        B = dev.to(torch.float64) * scales.double().repeat_interleave(128)[:m.ncols, None]
    else:
        dev = B
        B = B.double()
    dev = dev.cuda()
    sc = scales.cuda() if scales is not None else None
    C = torch.full((m.nrows, n), float("nan"), device="cuda")
    torch.cuda.synchronize()  # inputs made on torch's stream are complete
    p.spmm(dev.data_ptr(), n, n, dt, C.data_ptr(), n, sc.data_ptr() if sc is not None else None)
    torch.cuda.synchronize()
    ref, mag, terms = _reference(m, B)
    bound = (terms[:, None] + 3) * 2.0 ** -24 * mag
    off = np.abs(C.cpu().numpy() - ref) - bound
    assert not np.isnan(off).any()
    assert (off <= 0).all(), (dt, n, np.argwhere(off > 0)[:5])
