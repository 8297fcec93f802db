"""Single sweeps that start from the best candidate between long edges.

The first cap may only come from a candidate of the tour itself: a pair of edges
with a common end, the closing edge, or an entry no wave wrote would drop the
best move.  Sizes around the one from which it is used, around whole waves and
workgroups, and above one edge per wave turn; starts with long edges anywhere,
with ties, and without any improving move.
"""
import os

import numpy as np
import pytest

import logo2opt as L
import oracle_lib as O

pytestmark = pytest.mark.gpu
THREADS = min(16, os.cpu_count() or 1)


@pytest.mark.parametrize("n", [999, 1000, 1001, 1024, 1025, 1089, 4095, 4097, 16385, 65537, 70001])
@pytest.mark.parametrize("prune", [False, True])
def test_step_with_first_cap(n, prune):
    xy = O.gen_uniform(n, 10**6, n)
    ties = O.gen_uniform(n, 30, n)
    near = O.nn_tour(xy, 0) if n < 20000 else L.nn_tour(xy, 0)
    far = np.roll(near, n // 2)  # the long closing edge inside, another one closing
    for pts, tours in ((xy, [near, far, O.random_perm(n, 3)]), (ties, [O.random_perm(n, 4)])):
        with L.Context(L.coords_of(pts)) as ctx:
            ctx.set_pruning(prune)
            for t in tours:
                ok, move = O.step_fast(pts, t, THREADS)
                for _ in range(2):  # the slot's next instance takes over its record
                    assert ctx.step(t) == (move if ok else (0, 0, 0))


@pytest.mark.parametrize("metric", [0, 1, 2])
def test_step_without_a_move_and_after_searches(metric):
    n = 2000
    xy = O.gen_uniform(n, 10**5, 8)
    with L.Context(L.coords_of(xy), metric=metric) as ctx:
        start = O.random_perm(n, 5)
        for _ in range(2):
            out = ctx.optimize(start)
            assert ctx.step(out["route"]) == (0, 0, 0)
            ok, move = O.step(xy, start, THREADS, metric=metric)
            assert ctx.step(start) == move
            assert ctx.route_length(start) == L.host_route_length(L.coords_of(xy), start, metric)
            with pytest.raises(L.Logo2OptError):  # refused: the slot's record is cleared
                ctx.step(np.zeros(n, np.uint32))
            assert ctx.optimize(start)["length"] == out["length"]
