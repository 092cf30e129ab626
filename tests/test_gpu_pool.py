"""The device memory that a context keeps between its calls (GPU): results on
reused buffers equal those on fresh ones, over calls of growing and shrinking
size, with objects that outlive their call, and with two contexts in threads."""
import threading

import numpy as np
import pytest
import torch

import vnm

pytestmark = pytest.mark.gpu
SIZES = [(300, 4), (4096, 12), (900, 6), (5000, 9), (300, 4), (4096, 12)]


def product(ctx, p, n, B):
    C = torch.full((n, 64), float("nan"), device="cuda")
    torch.cuda.current_stream().synchronize()
    p.spmm(B.data_ptr(), 64, 64, vnm.DT_F32, C.data_ptr(), 64)
    torch.cuda.ExternalStream(ctx.stream).synchronize()
    return C.cpu().numpy()


def call(ctx, n, deg, keep):
    rng = np.random.default_rng(n)
    r = rng.integers(0, n, n * deg).astype(np.int32)
    c = rng.integers(0, n, n * deg).astype(np.int32)
    m = vnm.coo_from_tuples(n, n, r, c, rng.uniform(-1, 1, n * deg).astype(np.float32), 8)
    n = -(-n // 8) * 8  # the operand and the result have the padded rows
    B = torch.from_numpy(rng.standard_normal((n, 64)).astype(np.float32)).cuda()
    g = vnm.Graph(ctx, m, 8)
    g.lp_reorder(None, 2, mode=vnm.LP_EXHAUSTIVE, maxiter=3)
    p = g.pack(64, vnm.DT_F32)
    out = product(ctx, p, n, B)
    keep.append((g, p, n, B, out))
    return out, g.perm()


def series(ctx, out):
    keep = []
    out.extend(call(ctx, n, d, keep) for n, d in SIZES)
    for g, p, n, B, ref in keep[::-1]:  # objects still whole after the later calls
        assert np.array_equal(product(ctx, p, n, B), ref)


def test_reused_buffers():
    fresh = [call(vnm.Context(0), n, d, []) for n, d in SIZES]
    got = [[], []]
    ts = [threading.Thread(target=series, args=(vnm.Context(0), got[i])) for i in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for res in got:
        assert len(res) == len(fresh)
        for (a, pa), (b, pb) in zip(res, fresh):
            assert np.array_equal(a, b) and np.array_equal(pa, pb)


def test_trim_gives_idle_memory_back():
    ctx = vnm.Context(0)
    first = call(ctx, 65536, 16, [])  # its graph and packed matrix are gone
    torch.cuda.synchronize()
    idle = torch.cuda.mem_get_info()[0]
    ctx.trim()
    assert torch.cuda.mem_get_info()[0] >= idle + (32 << 20)
    again = call(ctx, 65536, 16, [])
    assert all(np.array_equal(a, b) for a, b in zip(first, again))


def test_batched_learned_reorder_on_reused_buffers():
    M, N = 8, 2
    rng = np.random.default_rng(8)
    coos = [vnm.gen_chung_lu(int(n), 2.1, 12.0, 40 + i, M=M) for i, n in enumerate(rng.integers(300, 9000, 12))]
    ctx = vnm.Context(0)
    model = vnm.LPModel(ctx, seed=1)
    fresh = vnm.Context(0)
    fresh_model = vnm.LPModel(fresh, seed=1)
    for order in (range(12), range(11, -1, -1), range(0, 12, 3)):
        for mode, m in ((vnm.LP_LEARNED, model), (vnm.LP_EXHAUSTIVE, None)):
            gs = [vnm.Graph(ctx, coos[i], M) for i in order]
            vnm.Graph.lp_reorder_batch(gs, m, N, mode=mode, topk=512, window=8, maxiter=4, seed=3)
            call(ctx, 900, 6, [])  # other calls take and give blocks of the same pool
            for i, g in zip(order, gs):
                alone = vnm.Graph(fresh, coos[i], M)
                alone.lp_reorder(fresh_model if m else None, N, mode=mode, topk=512, window=8, maxiter=4, seed=3)
                assert np.array_equal(g.perm(), alone.perm())
