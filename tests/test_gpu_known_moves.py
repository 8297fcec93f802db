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
        for sync in (1, 2, 3, 5, 64):
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


@pytest.mark.parametrize("n", [3, 4, 8, 63, 64, 65, 66, 129, 321, 799, 800, 801])
def test_one_workgroup_searches(n):
    """Sizes around the 32-edge blocks, the 64-edge pairs and the largest size
    that one workgroup takes, as a search, in slices, and as an ILS job."""
    xy = O.gen_uniform(n, 3000, n)
    r0 = O.random_perm(n, n + 2)
    r, Lo, moves, _, log = O.local_search(xy, r0, threads=THREADS)
    with L.Engine(max_slots=3) as e:
        co = L.coords_of(xy)
        s = e.add(co, r0, log_cap=4096)
        k = e.add(co, r0, log_cap=4096)
        e.run(max_steps=moves // 2, sync_every=4)
        assert e.result(s)["moves"] == moves // 2
        while e.run(max_steps=7, sync_every=4):
            pass
        for slot in (s, k):  # (the second one starts with the first)
            out = e.result(slot, n, log_cap=4096)
            assert out["length"] == Lo and out["sweeps"] == moves + 1
            np.testing.assert_array_equal(out["log"], log)
            assert out["route"].tolist() == r.tolist()
    if n >= 8:
        for kick in (0, 1):
            br, bl, hist, _ = O.ils(xy, r0, 9, 6, kick=("double_bridge", "reference")[kick], threads=THREADS)
            with L.Context(L.coords_of(xy)) as ctx:
                gr, gl, gh = ctx.ils(r0, 9, 6, kick)
            assert gl == bl and gh.tolist() == list(hist) and gr.tolist() == br.tolist()


def test_many_small_instances_and_chains():
    """More than 64 instances (four waves each) beside larger ones, and chains
    of one instance whose rounds alternate with the group's barrier."""
    rng = np.random.default_rng(4)
    jobs = [(int(n), int(s)) for n, s in zip(rng.integers(8, 900, 70), rng.integers(0, 1000, 70))] + [(1500, 5), (1300, 6)]
    with L.Engine(max_slots=80) as e:
        slots = []
        for n, s in jobs:
            xy = O.gen_uniform(n, 10**4, s)
            slots.append((e.add(L.coords_of(xy), O.nn_tour(xy, 0)), xy, n))
        assert e.run() == 0
        for slot, xy, n in slots:
            r, Lo, moves, _, _ = O.local_search(xy, O.nn_tour(xy, 0), threads=THREADS)
            out = e.result(slot, n)
            assert (out["length"], out["moves"]) == (Lo, moves) and out["route"].tolist() == r.tolist()
    xy = O.gen_uniform(500, 10**4, 3)
    r0 = O.random_perm(500, 4)
    want = O.ils_multistart(xy, r0, 11, 7, 5)
    with L.Context(L.coords_of(xy)) as ctx:
        got = ctx.ils_multistart(r0, 11, 7, 5)
    assert got[1] == want[1] and got[2].tolist() == list(want[2]) and got[0].tolist() == np.asarray(want[0]).tolist()
