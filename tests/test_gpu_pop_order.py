"""Pop orders by a wave a list (up to 4,096 lists) and by a thread a list (more)
are the same, ties included, for every list size and around the limit (GPU).
The thread's heap is the one that the host test holds against libstdc++."""
import numpy as np
import pytest

import vnm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 7, 8])
@pytest.mark.parametrize("distinct", [1, 5, 1000])
def test_wave_and_thread(M, distinct):
    rng = np.random.default_rng(M + 10 * distinct)
    sc = rng.integers(-distinct, distinct + 1, (4097, M * M, 2)).astype(np.int32)
    sc[1] = 2**31 - 1 - 2**30 - rng.integers(0, 2, (M * M, 2))  # gains near the type's ends, sums in range
    sc[2] = -(2**30) + rng.integers(0, 2, (M * M, 2))
    ctx = vnm.Context(0)
    threads = ctx.pq_pop_order(sc, M)  # 4,097 lists
    waves = ctx.pq_pop_order(sc[:4096], M)
    assert np.array_equal(threads[:4096], waves)
    assert np.array_equal(threads[4096:], ctx.pq_pop_order(sc[4096:], M))
    assert np.array_equal(np.sort(waves, axis=1), np.tile(np.arange(M * M), (4096, 1)))
