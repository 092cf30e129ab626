"""The SpMM's work items and column tiles at their edges (GPU).

Rows of every length around the item and block sizes (1 to 66 values, whole
chunks, chunks with a remainder, a hub row of more than 16 chunks), rows without
values before the first row, in runs of 8 and 9, after a cut row and at the end,
and column counts of one to eight 64-column groups, among them FP8 rows of an odd
number of those, at the width that the rule takes and at every other one.  Every
entry is kept (one per 4-column segment, V = 1), so the reference is the plain product
in FP64; an output of L terms in FP32 may be off by (L + 3) 2^-24 times the sum of the
terms' magnitudes (one rounding per FMA, one for the weight's scale, and the chunk
sums).
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


def _operand(m, dt, n):
    """(B on the device, its scales, B in FP64)."""
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
    return dev.cuda(), scales.cuda() if scales is not None else None, B


def _product(m, p, dt, n, dev, sc):
    C = torch.full((m.nrows, n), float("nan"), device="cuda")
    torch.cuda.synchronize()  # inputs made on torch's stream are complete
    p.spmm(dev.data_ptr(), n, n, dt, C.data_ptr(), n, sc.data_ptr() if sc is not None else None)
    torch.cuda.synchronize()
    return C.cpu().numpy()


@pytest.mark.parametrize("dt", [vnm.DT_F32, vnm.DT_BF16, vnm.DT_FP8])
@pytest.mark.parametrize("n", [64, 128, 192, 320, 512])
def test_items_and_tiles_at_their_edges(matrix, dt, n):
    m, g, p = matrix
    dev, sc, B = _operand(m, dt, n)
    C = _product(m, p, dt, n, dev, sc)
    ref, mag, terms = _reference(m, B)
    bound = (terms[:, None] + 3) * 2.0 ** -24 * mag
    off = np.abs(C - ref) - bound
    assert not np.isnan(off).any()
    assert (off <= 0).all(), (dt, n, np.argwhere(off > 0)[:5])


@pytest.mark.parametrize("dt,size", [(vnm.DT_F32, 4), (vnm.DT_BF16, 2), (vnm.DT_FP8, 1)])
@pytest.mark.parametrize("n", [64, 192, 512, 1024])
def test_every_width_gives_the_rule_s_bits(matrix, dt, size, n):
    m, g, p = matrix
    dev, sc, _ = _operand(m, dt, n)
    p.set_shape(dt, n, 0)
    C = _product(m, p, dt, n, dev, sc)
    rule = p.get_shape(dt, n)
    widths = [v for v in (1, 2, 4, 8, 16) if n % (64 * v) == 0 and 2 <= v * size <= 16] or [1]
    assert rule in widths
    assert n // (64 * rule) <= 8 or rule == widths[-1]  # no more tiles than XCDs where a width allows
    for v in widths:
        p.set_shape(dt, n, v)
        assert p.get_shape(dt, n) == v
        assert np.array_equal(_product(m, p, dt, n, dev, sc), C), v
    # the batch takes the same widths, two matrices of a unit list
    out = [torch.full((m.nrows, n), float("nan"), device="cuda") for _ in range(2)]
    for v in [0] + widths:
        b = vnm.Batch(g.ctx, [p, p], [dev.data_ptr()] * 2, [n] * 2, n, dt, [c.data_ptr() for c in out], [n] * 2,
                      b_scales=[sc.data_ptr()] * 2 if sc is not None else None, cols_per_lane=v)
        for c in out:
            c.fill_(float("nan"))
        torch.cuda.synchronize()
        b.run()
        torch.cuda.synchronize()
        assert all(np.array_equal(c.cpu().numpy(), C) for c in out), v
        b.close()
    p.set_shape(dt, n, 0)
    for v in {1, 2, 4, 8, 16, 3} - set(widths):  # what no product takes stays refused
        with pytest.raises(vnm.VnmError):
            p.set_shape(dt, n, v)


@pytest.mark.parametrize("cut", [False, True])
def test_width_for_a_far_operand(cut):
    """512 MiB of B: the widest tile, unless many values lie in cut rows."""
    rng = np.random.default_rng(6)
    R, n = 1 << 20, 128
    r, c = rng.integers(0, R, 3000), rng.integers(0, R, 3000)
    if cut:
        r, c = np.r_[r, np.full(300, 7)], np.r_[c, rng.choice(R // 4, 300, replace=False) * 4]
    m = vnm.coo_from_tuples(R, R, r.astype(np.int32), c.astype(np.int32), rng.normal(size=len(r)).astype(np.float32), 4)
    p = vnm.Graph(vnm.Context(0), m, 4).pack(1, vnm.DT_F32)
    B = torch.randn(R, n, generator=torch.Generator(device="cuda").manual_seed(2), device="cuda")
    C = _product(m, p, vnm.DT_F32, n, B, None)
    assert p.get_shape(vnm.DT_F32, n) == (1 if cut else 2)
    for v in (1, 2):
        p.set_shape(vnm.DT_F32, n, v)
        assert np.array_equal(_product(m, p, vnm.DT_F32, n, B, None), C)
