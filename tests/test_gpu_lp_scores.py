"""One iteration of the learned reorder with scores that are not ordinary numbers
(GPU): every donor score the NaN of all ones, pair scores that are infinite or NaN, and
plain ones.  The iteration is restated here from its rules --
a donor and an acceptor per segment by strict comparisons in bit order, donors and
acceptors ranked by the order of the scores' bits, a donor's window walked entry by
entry, the segment-disjoint walk over the exact gains -- and gives the relabel."""
import numpy as np
import pytest

import vnm

pytestmark = pytest.mark.gpu
N, M, TOPK, WINDOW = 2, 8, 24, 16
WH, BH = 18624, 22720  # the head's weights and biases


def _ordered(f):
    """Integers that order as the scores are ranked (bits of floats, sign folded)."""
    u = int(np.float32(f).view(np.uint32))
    return u ^ 0xFFFFFFFF if u & 0x80000000 else u | 0x80000000


def _pair(yu, yv):
    s = np.float32(yu[0] + yv[1])
    for t in range(16):  # a fused multiply-add a term
        s = np.float32(np.float64(yu[2 + t]) * np.float64(yv[18 + t]) + np.float64(s))
    return s


def _iteration(g, m, Y):
    """perm after one iteration over the unlabelled graph."""
    R, ns = m.nrows, m.nrows // M
    A = np.zeros((R, R), bool)
    A[m.row[m.val != 0], m.col[m.val != 0]] = True
    full = A.reshape(R, ns, M).sum(2)  # a row's ones in each segment
    donors, acceptors = [], []
    for s in range(ns):
        invalid = (full[:, s] > N).any()
        bd = ba = None
        for b in range(M):
            u = s * M + b
            if invalid and (A[:, u] & (full[:, s] == N + 1)).any() and (bd is None or Y[u, 0] > Y[bd, 0]):
                bd = u
            if ba is None or Y[u, 1] > Y[ba, 1]:
                ba = u
        if bd is not None:
            donors.append((-_ordered(Y[bd, 0]), s, bd))
        acceptors.append((-_ordered(Y[ba, 1]), s, ba))
    donors.sort()
    acceptors.sort()
    nd = min(TOPK, len(donors))
    assert nd > 1
    stride = max(1, ns // nd)
    cand, nans = [], 0
    for i in range(nd):
        _, p, u = donors[i]
        best = None
        for w in range(WINDOW):
            _, q, v = acceptors[(i * stride + w) % ns]
            if q == p:
                continue
            sc = _pair(Y[u], Y[v])
            nans += bool(np.isnan(sc))
            if best is None or sc > best[0]:
                best = (sc, q)
        cand.append((p, best[1]))
    gains = g.pair_score(N, [p for p, _ in cand], [q for _, q in cand]).reshape(nd, M * M, 2).astype(np.int64)
    pick = []
    for i in range(nd):
        lg, rg = gains[i, :, 0], gains[i, :, 1]
        j = min(range(M * M), key=lambda e: (-(lg[e] + rg[e]), -rg[e], e))
        pick.append((int(-(lg[j] + rg[j])), i, j))
    perm, used = np.arange(R, dtype=np.int32), set()
    for neg, i, j in sorted(pick):
        p, q = cand[i]
        if neg >= 0 or p in used or q in used:
            continue
        used |= {p, q}
        a, b = p * M + j // M, q * M + j % M
        perm[a], perm[b] = b, a
    return perm, len(used) // 2, nans


@pytest.mark.parametrize("kind", ["plain", "nan", "mixed"])
def test_iteration(kind):
    rng = np.random.default_rng(29)
    R = 512
    r, c = rng.integers(0, R, 9000), rng.integers(0, R, 9000)
    # segments without a row of N + 1 ones, and so without a donor, among the others
    keep = (c // M) % 5 != 0
    m = vnm.coo_from_tuples(R, R, r[keep], c[keep], np.ones(int(keep.sum()), np.float32), M)
    ctx = vnm.Context(0)
    P = vnm.LPModel(ctx, seed=3).params()
    head = P[WH:BH].reshape(64, 64)
    head[:, :34] *= 4
    if kind == "nan":
        P[BH:BH + 1] = np.array([0xFFFFFFFF], np.uint32).view(np.float32)
    elif kind == "mixed":  # P1 Q1 + P2 Q2 with P infinite: NaN where the signs differ
        P[BH + 3:BH + 5] = np.inf
    lm = vnm.LPModel(ctx, params=P)
    g = vnm.Graph(ctx, m, M)
    Y = lm.forward(g, N, bf16=True)
    with np.errstate(all="ignore"):
        perm, swaps, nans = _iteration(g, m, Y)
    assert swaps > 0 and (nans > 0) == (kind != "plain")
    st = g.lp_reorder(lm, N, mode=vnm.LP_LEARNED, topk=TOPK, window=WINDOW, maxiter=1)
    assert st.swaps == swaps
    assert np.array_equal(g.perm(), perm)
