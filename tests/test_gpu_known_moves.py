"""Improving moves carried from one tour to the next.

A sweep starts from the best candidate of earlier sweeps that the last move
left valid, at its mapped positions.  A wrong mapping (a side mixed up, a
removed edge kept, a stale entry of the slot's former instance) would publish a
move that does not exist and change the move log.  Instances with few distinct
edge lengths make almost every selection a tie, so the mapped positions decide.
"""
import os

import numpy as np
import pytest

import logo2opt as L
import oracle_lib as O

pytestmark = pytest.mark.gpu
THREADS = min(16, os.cpu_count() or 1)


@pytest.mark.parametrize("n,side,metric", [(5, 4, 0), (8, 3, 1), (64, 5, 0), (257, 8, 2), (600, 12, 0), (1025, 40, 1),
                                           (2050, 10**6, 0)])
@pytest.mark.parametrize("prune", [False, True])
def test_move_log_with_ties(n, side, metric, prune):
    xy = O.gen_uniform(n, side, 7 * n + side)
    r0 = O.random_perm(n, n + 1)
    r, Lo, moves, sweeps, log = O.local_search(xy, r0, threads=THREADS, metric=metric)
    with L.Context(L.coords_of(xy), metric=metric) as ctx:
        ctx.set_pruning(prune)
        for sync in (1, 64):
            out = ctx.optimize(r0, log_cap=1 << 14, sync_every=sync)
            np.testing.assert_array_equal(out["log"], log)
            assert out["length"] == Lo and out["route"].tolist() == r.tolist()


def test_slot_reuse_after_removal_mid_search():
    """A search removed half-way leaves nothing to the slot's next instance."""
    n = 500
    with L.Engine(max_slots=1) as e:
        for k in range(4):
            xy = O.gen_uniform(n, 10**4 if k % 2 else 30, 50 + k)
            r0 = O.random_perm(n, 60 + k)
            co = L.coords_of(xy)
            s = e.add(co, r0)
            e.run(max_steps=40 + 30 * k, sync_every=8)
            e.remove(s)
            m = 300 + k
            xy = O.gen_uniform(m, 10**4, 70 + k)
            r1 = O.nn_tour(xy, 0)
            r, Lo, moves, _, log = O.local_search(xy, r1, threads=THREADS)
            s = e.add(L.coords_of(xy), r1, log_cap=4096)
            e.run()
            out = e.result(s, m, log_cap=4096)
            np.testing.assert_array_equal(out["log"], log)
            assert out["length"] == Lo and out["route"].tolist() == r.tolist()
            e.remove(s)
