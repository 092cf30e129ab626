"""The GCN layer's X W at its tile rules (GPU): 64-row tiles, 128-row tiles with a
workgroup a panel and with all panels in one, a K of one stage, of half steps and
of two stages, rows short of a tile, X at a pitch and W at 2-byte alignment.  A
has a one in every row, so Y is a row of X W rounded to BF16, plus the bias: half a
BF16 ulp of the FP64 product and FP32's accumulation of K terms."""
import numpy as np
import pytest
import torch

import vnm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [8, 1000, 16408, 33000])
@pytest.mark.parametrize("K,N,pad", [(16, 64, 0), (48, 192, 4), (256, 128, 8), (272, 64, 0), (528, 128, 4)])
def test_tiles(R, K, N, pad):
    rng = np.random.default_rng(R + K)
    col = rng.permutation(R).astype(np.int32)
    ctx = vnm.Context(0)
    g = vnm.Graph(ctx, vnm.coo_from_tuples(R, R, np.arange(R, dtype=np.int32), col, np.ones(R, np.float32), 8), 8)
    p = g.pack(1, vnm.DT_BF16)
    X = torch.from_numpy(rng.standard_normal((R, K + pad)).astype(np.float32)).cuda().bfloat16()
    W = torch.from_numpy(rng.standard_normal(K * N + 1).astype(np.float32)).cuda().bfloat16()[1:].view(K, N)
    b = torch.from_numpy(rng.standard_normal(N).astype(np.float32)).cuda()
    Y = torch.full((R, N), float("nan"), device="cuda")
    torch.cuda.synchronize()
    p.gcn_layer(X.data_ptr(), K + pad, K, W.data_ptr(), N, Y.data_ptr(), N, b.data_ptr())
    torch.cuda.synchronize()
    x, w = X[:, :K].double().cpu(), W.double().cpu()
    H = (x @ w)[torch.from_numpy(col).long()]
    S = (x.abs() @ w.abs())[torch.from_numpy(col).long()]
    ref = H + b.double().cpu()
    tol = H.abs() * 2.0**-8 + (K + 2) * 2.0**-23 * S + ref.abs() * 2.0**-23
    assert ((Y.double().cpu() - ref).abs() <= tol).all()
