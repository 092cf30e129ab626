"""The greedy's choice of segments where there are more than a workgroup holds in
registers (4,096; GPU): few invalid segments, equal counts, counts that rise and fall
with the segment, and invalid segments that all fall to one thread.  Relabelled
matrix and stats of some rounds against the oracle, for every schedule."""
import numpy as np
import pytest

import oracle
import vnm

pytestmark = pytest.mark.gpu
N, M = 2, 8


def _counts(kind, nseg, rng):
    cnt = np.zeros(nseg, np.int64)
    if kind == "few":
        cnt[rng.choice(nseg, 5, replace=False)] = rng.integers(1, 4, 5)
    elif kind == "two":
        cnt[[nseg - 1, 4095]] = 2
    elif kind == "equal":
        cnt[rng.choice(nseg, nseg // 2, replace=False)] = 1
    elif kind == "rising":
        cnt[:] = np.arange(nseg) * 12 // nseg
    elif kind == "falling":
        cnt[:] = 12 - np.arange(nseg) * 12 // nseg
    else:  # one thread's segments, and a few others below them
        cnt[37::1024] = rng.integers(5, 9, len(cnt[37::1024]))
        cnt[rng.choice(nseg, 40, replace=False)] += 1
    return cnt


@pytest.mark.parametrize("nseg", [4096, 4097, 8200, 17000])
@pytest.mark.parametrize("kind", ["few", "two", "equal", "rising", "falling", "thread"])
def test_rounds(kind, nseg):
    rng = np.random.default_rng(nseg)
    cnt = _counts(kind, nseg, rng)
    R = nseg * M
    seg = np.repeat(np.arange(nseg), cnt)
    row = rng.permutation(R)[: len(seg)]
    col = np.stack([rng.permutation(M)[:3] for _ in range(64)])[rng.integers(0, 64, len(seg))] + seg[:, None] * M
    r, c = np.repeat(row, 3).astype(np.int32), col.ravel().astype(np.int32)
    m = vnm.coo_from_tuples(R, R, r, c, np.ones(len(r), np.float32), M)
    ctx = vnm.Context(0)
    for sched in (0, 1, 2, 3, 9):
        om = oracle.Matrix(m.nrows, m.ncols, m.row.copy(), m.col.copy(), m.val.copy())
        want = oracle.nm_reorder_sample(om, N, M, sched, 10, 12)
        g = vnm.Graph(ctx, m, M)
        got, _ = g.nm_trace(N, sched, 10, round_cap=12)
        assert got == list(want), sched
        out = g.download()
        assert np.array_equal(out.row, om.row) and np.array_equal(out.col, om.col), sched
        g.close()
