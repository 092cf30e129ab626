"""The values of a hybrid run's reload (GPU) against the text round trip itself
("%.2f", read back, "%.1e", read back): two-digit ties on both sides, all short
hundredths, signs, zeros, denormals, the limit of 2^24 and beyond."""
import numpy as np
import pytest

import vnm

pytestmark = pytest.mark.gpu


def _text(v):
    return np.float32(float("%.1e" % float("%.2f" % float(v))))


@pytest.mark.parametrize("long_values", [False, True])
def test_text_round_trip(long_values):
    rng = np.random.default_rng(3)
    v = [k / 100 for k in range(1, 2000)] + [k + 0.5 for k in range(100, 1000)]
    v += [1.05, 1.15, 1.25, 1.35, 9.95, 0.995, 99.5, 0.004999, 0.005, 1e-30, 1e-42, 16777215.0, 12500000.0, 1350.0]
    v += list(rng.uniform(-1, 1, 500)) + list(10.0 ** rng.uniform(-4, 7.2, 500))
    if long_values:
        v += [16777216.0, 3.05e8, 1.25e37, 3.4e38, -2.5e20]
    v = np.array(v, np.float32)
    v[::3] *= -1
    R = 64
    pos = rng.permutation(R * R)[: len(v)]
    m = vnm.coo_from_tuples(R, R, (pos // R).astype(np.int32), (pos % R).astype(np.int32), v, 8)
    g = vnm.Graph(vnm.Context(0), m, 8)
    kept = np.sort(m.val.copy())
    g.hybrid(2, 4, 1, 0)
    got = g.download().val
    want = np.sort(np.array([_text(x) for x in kept], np.float32))
    assert np.array_equal(np.sort(got), want)
