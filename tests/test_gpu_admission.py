"""Instances made on the device, and work lists kept between calls.

The device makes an admitted instance's ordered points and its length from the
cities and the tour; a slot's next instance of the same size keeps the work
lists of the last.  Everything is compared with the host's lengths and with the
oracle's searches, exactly.
"""
import os

import numpy as np
import pytest

import logo2opt as L
import oracle_lib as O

pytestmark = pytest.mark.gpu
THREADS = min(16, os.cpu_count() or 1)


@pytest.mark.parametrize("n", [3, 4, 5, 255, 256, 257, 1025, 65535, 65537, 140001])
@pytest.mark.parametrize("metric", [0, 1, 2])
def test_admitted_instance(n, metric):
    rng = np.random.default_rng(n + metric)
    xy = rng.integers(-(2**21), 2**21, 2 * n)  # moved to the origin, over the full range
    c = L.coords_of(xy)
    with L.Engine(max_slots=2) as e:
        s = []
        tours = [rng.permutation(n).astype(np.uint32) for _ in range(2)]
        for t in tours:
            s.append(e.add(c, t, metric=metric))
        for k in (1, 0):
            out = e.result(s[k], n)
            assert out["length"] == L.host_route_length(c, tours[k], metric)
            assert out["route"].tolist() == tours[k].tolist()


def test_many_admissions_before_a_run():
    """More waiting copies than the host buffer holds."""
    k, n = 40, 3001
    xy = O.gen_uniform(n, 10**5, 5)
    c = L.coords_of(xy)
    tours = [O.random_perm(n, q) for q in range(k)]
    with L.Engine(max_slots=k) as e:
        s = [e.add(c, t) for t in tours]
        for q in range(0, k, 2):
            e.remove(s[q])
        for q in range(1, k, 2):
            out = e.result(s[q], n)
            assert out["route"].tolist() == tours[q].tolist()
            assert out["length"] == L.host_route_length(c, tours[q], 0)


@pytest.mark.parametrize("n", [700, 3000])
def test_same_size_call_after_call(n):
    """Calls of every kind in turn on one context, each against the oracle."""
    xy = O.gen_uniform(n, 10**4, 1)
    with L.Context(L.coords_of(xy)) as ctx:
        for k in range(6):
            r0 = O.random_perm(n, 90 + k)
            r, Lo, moves, _, log = O.local_search(xy, r0, threads=THREADS)
            ctx.set_pruning(k % 3 == 2)
            before = ctx.stats()["moves"]
            out = ctx.optimize(r0, log_cap=1 << 14, sync_every=(1, 64, 64)[k % 3])
            np.testing.assert_array_equal(out["log"], log)
            assert out["length"] == Lo and out["route"].tolist() == r.tolist()
            assert ctx.stats()["moves"] - before == moves
            assert ctx.step(r0) == tuple(log[0])  # the search's first move
            assert ctx.step(r0, timing=True)[0] == tuple(log[0])
            ok, move = O.step(xy, r, THREADS)
            assert ctx.step(r) == (move if ok else (0, 0, 0))  # the optimum
            assert ctx.stats()["moves"] - before == moves
            b, best, rl = ctx.ils(r0, 5, 2)
            ob = O.ils(xy, r0, 5, 2, threads=THREADS)
            assert b.tolist() == ob[0].tolist() and best == ob[1]
