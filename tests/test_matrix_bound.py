"""The sweep's matrix test in exact integer arithmetic (numpy, no GPU).

Every candidate with gain <= cap has to pass |U - V|^2 - (E'_a + E'_b)^2 - 1 < 0
with the quantised coordinates and lengths of l2o_launch.h (set_quant,
quant_xy) and l2o_quant.h (quant_edge, edge_terms), and the terms have to fit
FP16 and FP32 exactly.
"""
import math

import numpy as np
import pytest

import oracle_lib as O

QR, QE = 640, 1830


def quantise(xy, metric):
    """(X, Y, qk, qm) in float32 arithmetic, as the library computes them."""
    f = np.float32
    x, y = xy[0::2].astype(np.int64), xy[1::2].astype(np.int64)
    x, y = x - x.min(), y - y.min()
    half = 0.5 * max(int(x.max()), int(y.max()))
    qs = f(4.0 if half * 4.0 <= 639.0 else 639.0 / half)
    kappa = math.sqrt(10.0) if metric == 2 else 1.0
    qk = np.nextafter(f(float(qs) * kappa), f(1e30))
    qm = f(1.02 + (0.5 * float(qs) if metric == 0 else 0.0))
    ox, oy = f(-0.5 * float(x.max()) * float(qs)), f(-0.5 * float(y.max()) * float(qs))
    X = (x.astype(f) * qs + ox + f(1024.5)).astype(np.int64) - 1024
    Y = (y.astype(f) * qs + oy + f(1024.5)).astype(np.int64) - 1024
    return x, y, X, Y, qk, qm


@pytest.mark.parametrize("metric", [0, 1, 2])
@pytest.mark.parametrize("side", [2, 30, 700, 10**4, 10**6, 2**22 - 1])
@pytest.mark.parametrize("start", ["random", "nn"])
def test_no_winning_candidate_is_dropped(metric, side, start):
    n = 180
    xy = O.gen_uniform(n, side, side % 1000 + metric)
    t = O.random_perm(n, 3) if start == "random" else O.nn_tour(xy, 0)
    x, y, X, Y, qk, qm = quantise(xy, metric)
    x, y, X, Y = (v[t.astype(np.int64)] for v in (x, y, X, Y))
    assert max(np.abs(X).max(), np.abs(Y).max()) <= QR

    def dist(dx, dy):
        s = (dx * dx + dy * dy).astype(np.float64)
        r = np.sqrt(s if metric != 2 else s / 10.0)
        return (np.floor(r + 0.5) if metric == 0 else np.ceil(r)).astype(np.int64)

    D = dist(np.diff(x), np.diff(y))                       # edge k -> k+1
    E = np.ceil((D.astype(np.float64) * float(qk) + float(qm)).astype(np.float32)).astype(np.int64)
    assert E.max() <= QE and E.min() >= 1
    U = X[:-1] ** 2 + Y[:-1] ** 2 + X[1:] ** 2 + Y[1:] ** 2
    a, b = np.triu_indices(n - 1, 2)
    G = dist(x[a] - x[b], y[a] - y[b]) + dist(x[a + 1] - x[b + 1], y[a + 1] - y[b + 1]) - D[a] - D[b]
    dist2 = ((X[a] - X[b]) ** 2 + (Y[a] - Y[b]) ** 2 + (X[a + 1] - X[b + 1]) ** 2 + (Y[a + 1] - Y[b + 1]) ** 2)
    assert dist2.tolist() == (U[a] + U[b] - 2 * (X[a] * X[b] + Y[a] * Y[b] + X[a + 1] * X[b + 1] +
                                                 Y[a + 1] * Y[b + 1])).tolist()
    best = int(min(G.min(), -1))
    for cap in sorted({-1, best, best // 2, best // 10 or -1}):
        hc = max(math.floor(np.float32(-cap) * np.float32(qk * np.float32(0.49999)) - np.float32(0.01)), 0)
        e = np.maximum(E - hc, 0)
        win = G <= cap
        acc = dist2 - (e[a] + e[b]) ** 2 - 1
        assert (acc[win] < 0).all()
        # exactness: FP16 terms of at most 2048, sums of positive and of negative terms below 2^24
        N = U - e ** 2
        Nh = N // 2048
        assert e.max() <= QE and np.abs(Nh).max() <= 2048
        worst = 8 * QR * QR + 4 * QE * QE
        assert worst < 2 ** 24
