"""The proposer's neighbour sums at the list lengths where its aggregation
changes path (GPU): empty, 1 to 17, around 64 (four lists to a wave), around 1,024
(one wave), and lists cut into two and three chunks -- as columns for the forward
pass and as rows for the backward one.  Head, loss and gradient against the
FP64 oracle at the FP32 path's bars (1e-5 of the result's norm, 1e-4 for the gradient)."""
import numpy as np
import pytest

import oracle
import vnm

pytestmark = pytest.mark.gpu
N, M = 2, 8


@pytest.mark.parametrize("transposed", [False, True])
def test_list_lengths(transposed):
    rng = np.random.default_rng(17)
    R = 2304
    lens = list(range(0, 18)) + [31, 32, 33, 63, 64, 65, 66, 127, 128, 129, 1023, 1024, 1025, 2047, 2049, 2300]
    c = np.concatenate([np.full(n, 5 * i + 3) for i, n in enumerate(lens)]).astype(np.int32)
    r = np.concatenate([np.sort(rng.choice(R, n, replace=False)) for n in lens]).astype(np.int32)
    if transposed:
        r, c = c, r
    m = vnm.coo_from_tuples(R, R, r, c, rng.uniform(0.1, 1, len(r)).astype(np.float32), M)
    ctx = vnm.Context(0)
    g = vnm.Graph(ctx, m, M)
    P = vnm.LPModel(ctx, seed=5).params()
    P[18624:22720].reshape(64, 64)[:, :34] *= 4  # a head that weighs in the loss
    lm = vnm.LPModel(ctx, params=P)
    pairs = rng.integers(0, R, (300, 2)).astype(np.int32)
    target = rng.normal(0, 1, 300)
    om = oracle.Matrix(m.nrows, m.ncols, m.row.copy(), m.col.copy(), m.val.copy())
    loss, grad, head = oracle.lp_loss_grad(om, N, M, P.astype(np.float64), pairs, target)
    Y = lm.forward(g, N, bf16=False)
    assert np.linalg.norm(Y - head) < 1e-5 * np.linalg.norm(head)
    got_loss, got = lm.loss_grad(g, N, pairs, target, bf16=False)
    assert abs(got_loss - loss) < 1e-5 * abs(loss)
    assert np.linalg.norm(got - grad) < 1e-4 * np.linalg.norm(grad)
