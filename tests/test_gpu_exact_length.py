"""The kernels' FP64-free edge length at its breakpoints.

Tours that go back and forth between the origin and points whose squared
distance lies at or next to k^2, k^2 + k and 10 k^2 (the breakpoints of the
three metrics), over the whole coordinate range, measured by the device and by
the host's integer-checked FP64 version.
"""
import numpy as np
import pytest

import logo2opt as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("metric", [L.METRIC_EUC_2D, L.METRIC_CEIL_2D, L.METRIC_ATT])
@pytest.mark.parametrize("hi", [64, 3000, 2**16, 2**20, 2**22 - 1])
def test_lengths_at_breakpoints(metric, hi):
    rng = np.random.default_rng(hi + metric)
    m = 20000
    k = rng.integers(0, hi, m)
    kind = np.arange(m) % 4
    s = np.where(kind == 0, k * k, np.where(kind == 1, k * k + k, np.where(kind == 2, 10 * (k * k // 10), k * k)))
    # x near the root, y makes up the rest as far as a square can (off by up to 2 y)
    x = np.minimum(np.floor(np.sqrt(s)).astype(np.int64), hi)
    x = np.maximum(x - rng.integers(0, 3, m) * (kind != 0), 0)
    y = np.floor(np.sqrt(np.maximum(s - x * x, 0))).astype(np.int64) + (kind == 3)
    y = np.minimum(y, hi)
    n = 2 * m
    px = np.zeros(n, np.float32)
    py = np.zeros(n, np.float32)
    px[1::2], py[1::2] = x, y
    px[1], py[1] = hi, hi  # the full span
    c = L.float_coords(px, py)
    with L.Context(c, n=n, metric=metric) as ctx:
        t = np.arange(n, dtype=np.uint32)
        assert ctx.route_length(t) == L.host_route_length(c, t, metric)
        for seed in range(3):  # any pairs of the points
            t = np.random.default_rng(seed).permutation(n).astype(np.uint32)
            assert ctx.route_length(t) == L.host_route_length(c, t, metric)
        # every edge by itself: the lengths of short tours through the origin
        for a in (1, 3, 5, 7, 9, 11, 13, 15):
            q = np.array([0, a], np.uint32)
            t = np.concatenate([q, np.setdiff1d(np.arange(n, dtype=np.uint32), q)])
            assert ctx.route_length(t) == L.host_route_length(c, t, metric)
