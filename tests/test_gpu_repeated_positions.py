"""Packing a graph whose positions repeat.

The allpairs schedules in compat mode relabel by a table that is not a
permutation where a node is swapped twice in a round (reorder/reorder.h:1194-1197):
positions merge, and the graph goes on with their entries side by side.  A row
of a block then keeps two entries of one column, so the kept values are more than
the retained positions, and the packed value stream has to hold them all.
"""
import numpy as np
import pytest

import oracle
import vnm

N, M = 2, 4
CASES = [(10, 4000, 5, 4), (11, 8000, 5, 5), (12, 30000, 3, 6), (12, 30000, 3, 7)]


def _merged(case):
    scale, edges, seed, sched = case
    m = vnm.gen_rmat(scale, edges, seed, M=M)
    om = oracle.Matrix(m.nrows, m.ncols, m.row.copy(), m.col.copy(), m.val.copy())
    _, overwrites = oracle.allpairs_reorder(om, N, sched, clean=False)
    assert overwrites > 0
    return m, om


def _row_entries(om):
    """(kept values, row entries, nonzero entries) of the matrix packed at V = 1,
    M = 4: every column is selected, and a row of a block keeps two entries."""
    live = om.val != 0
    _, per = np.unique(om.row[live].astype(np.int64) * (om.ncols // M + 1) + om.col[live] // M, return_counts=True)
    return int(np.minimum(per, 2).sum()), len(per), int(live.sum())


@pytest.mark.parametrize("case", CASES)
def test_values_outnumber_positions(case):
    """On the CPU: the cases have more values than positions, and no more than the
    stream is sized for."""
    _, om = _merged(case)
    values, entries, nonzero = _row_entries(om)
    retained = oracle.retained_nnz(om, 1, N, M)
    assert values > retained
    assert values <= min(nonzero, 2 * entries)


@pytest.mark.gpu
@pytest.mark.parametrize("V", [1, 16])
@pytest.mark.parametrize("case", CASES)
def test_product_of_merged_positions(case, V):
    torch = pytest.importorskip("torch")
    m, om = _merged(case)
    ctx = vnm.Context(0)
    g = vnm.Graph(ctx, m, M)
    g.nm_reorder_allpairs(N, case[3], clean=False)
    got = g.download()
    assert np.array_equal(got.row, om.row) and np.array_equal(got.col, om.col)
    p = g.pack(V, vnm.DT_F32)
    info = p.info()
    stored = (info.spmm_bytes - 16 * info.items) // 8  # 8 bytes a value, 16 a work item
    if V == 1:
        assert stored == _row_entries(om)[0]
    assert info.retained_nnz == oracle.retained_nnz(om, V, N, M)
    assert stored > info.retained_nnz
    B = vnm.gen_normal(9, (m.ncols, 64))
    Bd = torch.from_numpy(B).cuda()
    C = torch.full((m.nrows, 64), float("nan"), device="cuda")
    torch.cuda.synchronize()
    p.spmm(Bd.data_ptr(), 64, 64, vnm.DT_F32, C.data_ptr(), 64)
    torch.cuda.synchronize()
    ref = oracle.spmm_vnm_f64(om, V, M, B)
    # FP32 sums of a row's terms: the FP32 bar of the other products
    assert np.abs(C.cpu().numpy() - ref).max() < 1e-5 * np.abs(ref).max()
