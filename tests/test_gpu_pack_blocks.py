"""Packing where the blocks' grid (segments x V-row blocks) has 2^34 places (GPU): a
block is told from one 2^32 places away, in the row entries and in the sparse-MFMA
part.  Every entry is kept (few per row and segment), so the product is the plain
one in FP64; FP32 sums of at most 6 terms, BF16 operands taken as stored."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import vnm  # noqa: E402

pytestmark = pytest.mark.gpu
M, n = 4, 64


@pytest.mark.parametrize("log_rows,V,dtype,dense_min",
                         [(18, 1, vnm.DT_F32, 0), (20, 16, vnm.DT_BF16, 0), (20, 16, vnm.DT_BF16, 2)])
def test_far_blocks(log_rows, V, dtype, dense_min):
    rng = np.random.default_rng(log_rows)
    R = 1 << log_rows
    nseg, nblk = R // M, R // V
    assert nseg * nblk == 1 << 34
    step = (1 << 32) // nblk  # segments this far apart are 2^32 places apart
    rows = np.unique(rng.integers(0, R, 40))
    r, c = [], []
    for row in rows:
        seg = rng.integers(0, step)
        for k in range(3):  # the same place modulo 2^32, two of the four columns
            cols = (seg + k * step) * M + rng.choice(M, 2, replace=False)
            r += [row] * 2
            c += list(cols)
    v = rng.uniform(0.5, 2, len(r)).astype(np.float32)
    if dtype == vnm.DT_BF16:
        v = torch.from_numpy(v).bfloat16().float().numpy()
    m = vnm.coo_from_tuples(R, R, np.array(r, np.int32), np.array(c, np.int32), v, M)
    g = vnm.Graph(vnm.Context(0), m, M)
    p = g.pack(V, dtype, dense_min)
    info = p.info()
    assert info.retained_nnz == len(r)
    assert info.nblocks == len(np.unique(m.row.astype(np.int64) // V * nseg + m.col // M))
    assert (info.dense_blocks > 0) == (dense_min > 0)
    gen = torch.Generator(device="cuda").manual_seed(5)
    B = torch.randn(R, n, generator=gen, device="cuda")
    B = B.bfloat16() if dtype == vnm.DT_BF16 else B
    C = torch.full((R, n), float("nan"), device="cuda")
    torch.cuda.synchronize()
    p.spmm(B.data_ptr(), n, n, dtype, C.data_ptr(), n)
    torch.cuda.synchronize()
    want = np.zeros((len(rows), n))
    mag = np.zeros((len(rows), n))
    at = np.searchsorted(rows, m.row)
    Bc = B[torch.from_numpy(m.col.astype(np.int64)).cuda()].double().cpu().numpy()
    np.add.at(want, at, m.val.astype(np.float64)[:, None] * Bc)
    np.add.at(mag, at, m.val.astype(np.float64)[:, None] * np.abs(Bc))
    got = C[torch.from_numpy(rows).cuda()].double().cpu().numpy()
    assert (np.abs(got - want) <= 9 * 2.0 ** -24 * mag).all()
    C[torch.from_numpy(rows).cuda()] = 0
    assert (C == 0).all()
