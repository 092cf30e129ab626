"""The radix sort at the edges of its launch plans (GPU): one workgroup up to
4,096 keys, 1,024-key tiles up to 16,384, 4,096-key tiles in fused passes up to
65,536, three launches per pass above.  The order is numpy's stable argsort of
the low end_bit bits; widths around whole 8-bit passes and one-bit last digits.
The key-range and two-field sorts are exercised through the callers whose results
are pinned to the oracle (VENOM, packing, the proposer)."""
import numpy as np
import pytest

import vnm

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n", [1023, 1025, 4098, 5120, 5121, 16383, 65536, 65537, 69633])
@pytest.mark.parametrize("end_bit", [1, 9, 16, 33, 64])
def test_sort_at_plan_edges(n, end_bit):
    ctx = vnm.Context(0)
    rng = np.random.default_rng(n + end_bit)
    keys = rng.integers(0, 2 ** 63, n, dtype=np.int64).view(np.uint64) & np.uint64(0xF0F0F0F30F0F0F0F)
    mask = np.uint64((1 << end_bit) - 1) if end_bit < 64 else np.uint64(2 ** 64 - 1)
    order = np.argsort(keys & mask, kind="stable")
    kin = torch.from_numpy(keys.view(np.int64)).cuda()
    vin = torch.arange(n, dtype=torch.int32, device="cuda")
    kout, k2, vout = torch.empty_like(kin), torch.empty_like(kin), torch.empty_like(vin)
    torch.cuda.synchronize()  # inputs made on torch's stream are complete
    ctx.sort_pairs(kin.data_ptr(), kout.data_ptr(), n, end_bit, vin.data_ptr(), vout.data_ptr())
    ctx.sort_pairs(kin.data_ptr(), k2.data_ptr(), n, end_bit)
    torch.cuda.synchronize()
    assert np.array_equal(kout.cpu().numpy().view(np.uint64), keys[order])
    assert np.array_equal(k2.cpu().numpy().view(np.uint64), keys[order])
    assert np.array_equal(vout.cpu().numpy(), order.astype(np.int32))
