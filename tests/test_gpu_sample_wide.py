"""Sampling whose kept candidates do not fit the pick kernel's LDS, by counting: where the counting can go wrong (a
bucket that needs its second and third level, sums that cross in the last bucket and go to the whole-row sort, more
equal weights than fit, floors that cut a bucket, the longest row it takes and the first it does not), against the
oracle with the same draws. A token may differ only where the oracle's margin to a running-sum boundary is below 1e-6 of
the total (tests/test_gpu_rows.py)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rows_of(kind, n, rng):
    if kind == "spread":    # 30 octaves: the last bucket holds most weights
        return rng.uniform(-40, 0, (2, n)).astype(np.float32)
    if kind == "narrow":    # one bucket of the top level holds nearly all: second level
        return (1 + rng.random((2, n)) * 0.05).astype(np.float32)
    if kind == "needle":    # and of the second: third level
        return (1 + rng.random((2, n)) * 2e-5).astype(np.float32)
    if kind == "equal":     # more equal weights than fit: the whole-row sort
        return np.repeat(np.float32([[0.5], [-3.0]]), n, axis=1)
    return (rng.standard_normal((2, n)) * 2).astype(np.float32)


CASES = [("spread", 20000, dict(top_p=0.9999999)), ("spread", 60000, dict(min_p=1e-9)), ("spread", 60000, dict(top_p=0.9)),
         ("narrow", 30000, dict(top_p=0.5)), ("narrow", 30000, dict(top_p=0.9, min_p=0.97)),
         ("needle", 30000, dict(top_p=0.7)), ("equal", 10000, dict(top_p=0.6)), ("normal", 50257, dict(min_p=0.001)),
         ("normal", 50257, dict(top_p=0.999, min_p=0.001)), ("normal", 4097, dict(top_p=0.99999)),
         ("normal", (1 << 20) - 1, dict(top_p=0.95)), ("normal", 1 << 20, dict(top_p=0.95))]


@pytest.mark.parametrize("kind,n,params", CASES)
def test_sums_over_many_candidates(hip, orc, kind, n, params):
    rng = np.random.default_rng(n)
    x = rows_of(kind, n, rng)
    dx, dout = hip.array(x), hip.array(shape=(2,), dtype=np.int32)
    draws = [0.0, 0.3, 1 - 2.0 ** -53] if n < 1 << 19 else [0.4]
    for first in draws:
        u = np.array([first, rng.random()])
        hip.sample(dx, 2, n, u, dout, temperature=1.0, **params)
        got = dout.numpy()
        want, margin = orc.sample(x, u, temperature=1.0, **params)
        for r in range(2):
            assert got[r] == want[r] or margin[r] < 1e-6, (r, int(got[r]), int(want[r]), float(margin[r]))
    dx.free()
    dout.free()
