"""The small-world step (its stages in one workgroup's kernels, the block solve
with bodies in LDS and rows in registers) against a launch per stage and
colour (schedule field tailColours 0), bit for bit.

Sizes around where the path or its layout changes: below and beyond the rows
that lanes hold in registers (1024 with 256 lanes, 2048 with 512; 768 and 1536
with joints), the largest number of bodies in LDS and one beyond it, worlds
that start with more new pairs than the LDS sort takes, every joint type, a
body in more contacts than there are colours (the overflow colour), islands
that sleep, contacts that end, sub-worlds, a learned start, few iterations.
Larger worlds go to the team solve (the workgroups of one XCD with a barrier
between colours), with full and with small teams.
"""
import ctypes
import os
import sys
import threading

import numpy as np
import pytest

import engines as E

sys.path.insert(0, os.path.join(E.ROOT, "oracle"))
import mlp_ref as M  # noqa: E402

pytestmark = pytest.mark.gpu

BODY = np.dtype([
    ("type", "<i4"), ("flags", "<i4"), ("xf", "<f4", 4), ("lc", "<f4", 2), ("c0", "<f4", 2), ("a0", "<f4"),
    ("c", "<f4", 2), ("a", "<f4"), ("rest", "<f4", 12),
])
assert BODY.itemsize == 104
PROFILE = np.dtype([("name", "S24"), ("launches", "<i4"), ("pad", "<i4"), ("ms", "<f8")])


def a_launch_per_colour(w):
    ctx = w.device_context()
    lib = E.b2g_lib()
    sched = np.zeros(1, E.SCHEDULE)
    E.b2g_check(lib, ctx, lib.b2g_get_schedule(ctx, E.ptr(sched)))
    sched["tailColours"] = 0
    E.b2g_check(lib, ctx, lib.b2g_set_schedule(ctx, E.ptr(sched)))


def state(w):
    meta, man = w.contacts()
    st = w.stats()
    return (w.bodies().view(np.uint32), meta, E.manifold_bits(man),
            [int(st[k]) for k in ("contacts", "constraints", "points", "colours", "colouringRounds", "newPairs",
                                  "positionIterations", "beginEvents", "endEvents", "queries")],
            float(st["minSeparation"]), w.fat_aabbs().tobytes())


def run(w, per_colour, steps, vel=8, pos=3):
    try:
        if per_colour:
            a_launch_per_colour(w)
        out = []
        for _ in range(3):
            w.step(steps // 3, vel=vel, pos=pos)
            out.append(state(w))
        return out
    finally:
        w.close()


def same(a, b):
    for x, y in zip(a, b):
        for u, v in zip(x, y):
            assert np.array_equal(u, v) if isinstance(u, np.ndarray) else u == v


@pytest.mark.parametrize("kind, n, seed, steps, sleep, vel, pos", [
    ("pyramid", 1, 0, 60, True, 8, 3), ("pyramid", 12, 0, 90, True, 8, 3), ("pyramid", 33, 0, 30, False, 8, 3),
    ("world", 64, 1, 240, True, 8, 3), ("world", 500, 2, 240, False, 8, 3), ("world", 1000, 3, 300, False, 6, 2),
    ("world", 1700, 4, 330, False, 8, 3), ("world", 3000, 5, 60, False, 8, 3), ("world", 4031, 5, 420, False, 8, 3),
    ("world", 4032, 5, 60, False, 8, 3), ("world", 300, 6, 240, False, 1, 0), ("world", 300, 6, 60, False, 0, 1),
    ("plank", 100, 0, 120, False, 8, 3), ("terrain", 150, 3, 150, True, 8, 3),
    ("chains", 30, 8, 120, True, 8, 3), ("pendulums", 40, 0, 90, False, 8, 3), ("distance", 20, 0, 60, False, 8, 3),
    ("ropes", 20, 0, 60, False, 8, 3), ("welds", 12, 0, 90, True, 8, 3), ("friction", 16, 0, 60, False, 8, 3),
    ("motor", 12, 0, 60, False, 8, 3), ("pulley", 8, 0, 60, False, 8, 3), ("mouse", 8, 0, 60, False, 8, 3),
    ("prismatic", 12, 0, 60, False, 8, 3), ("wheels", 6, 0, 90, False, 8, 3), ("gears", 4, 0, 60, False, 8, 3),
    # the team solve
    ("world", 4033, 8, 420, True, 8, 3), ("world", 6000, 9, 300, False, 6, 2), ("world", 13000, 10, 480, False, 8, 3),
    ("world", 5000, 11, 240, False, 2, 0), ("world", 5000, 11, 240, False, 0, 2), ("plank", 4100, 0, 9, False, 8, 3),
])
def test_equals_a_launch_per_colour(gpu, kind, n, seed, steps, sleep, vel, pos):
    a = run(gpu.world(kind, n, seed, sleep=sleep), False, steps, vel, pos)
    b = run(gpu.world(kind, n, seed, sleep=sleep), True, steps, vel, pos)
    same(a, b)


@pytest.mark.parametrize("kind, n, ccd", [("terrain", 60, True), ("bullets", 40, True), ("sensors", 30, False),
                                          ("oneway", 6, True), ("bullets", 130, True), ("terrain", 250, True),
                                          ("plank", 100, True), ("world", 700, True), ("world", 2300, True)])
def test_with_events_and_sensors(gpu, kind, n, ccd):
    same(run(gpu.world(kind, n, 2, ccd=ccd), False, 60), run(gpu.world(kind, n, 2, ccd=ccd), True, 60))


@pytest.mark.parametrize("kind, n_worlds, n, sleep", [("world", 9, 120, True), ("pendulums", 5, 7, False),
                                                      # the team solve, islands that sleep one by one
                                                      ("world", 20, 263, True), ("world", 20, 263, False)])
def test_sub_worlds(gpu, kind, n_worlds, n, sleep):
    same(run(E.World.worlds(gpu, kind, n_worlds, n, 4, sleep), False, 240),
         run(E.World.worlds(gpu, kind, n_worlds, n, 4, sleep), True, 240))


def learned(w, scope, seed):
    """A random network's start for every step: impulses of the size of a contact's."""
    lib, ctx = E.b2g_lib(), w.device_context()
    p = M.random_params(np.random.default_rng(seed))
    p["ystd"] = 0.05
    p["ymean"] = 0.0
    E.b2g_check(lib, ctx, lib.b2g_mlp_set_params(ctx, E.ptr(np.atleast_1d(p))))
    E.b2g_check(lib, ctx, lib.b2g_set_learned_scope(ctx, scope, 1))
    w.set_learned(True, 0.0)
    return w


@pytest.mark.parametrize("scope", [0, 1])
@pytest.mark.parametrize("n, steps", [(700, 240), (3000, 240), (6000, 300)])
def test_with_a_learned_start(gpu, n, steps, scope):
    """The network's impulses reach the rows that the block solve (two sizes)
    and the team solve hold."""
    a = learned(gpu.world("world", n, 3, sleep=False), scope, 5)
    b = learned(gpu.world("world", n, 3, sleep=False), scope, 5)
    same(run(a, False, steps), run(b, True, steps))
    plain = gpu.world("world", n, 3, sleep=False)
    plain.step(60)
    c = learned(gpu.world("world", n, 3, sleep=False), scope, 5)
    c.step(60)
    assert not np.array_equal(plain.bodies(), c.bodies()) and np.isfinite(c.bodies()).all()
    plain.close(); c.close()


@pytest.mark.parametrize("n, team", [(4033, 1), (9000, 1), (9000, 3), (13000, 5)])
def test_small_teams(gpu, n, team):
    """A team smaller than its constraints need reads those that its lanes
    cannot hold from memory in every pass, and turns the workgroups away that
    come once it is complete."""
    a = gpu.world("world", n, 8, sleep=False)
    ctx, lib = a.device_context(), E.b2g_lib()
    assert lib.b2g_set_team_size(ctx, 0) != 0 and lib.b2g_set_team_size(ctx, 17) != 0
    E.b2g_check(lib, ctx, lib.b2g_set_team_size(ctx, team))
    same(run(a, False, 300), run(gpu.world("world", n, 8, sleep=False), True, 300))


def launches(w, steps):
    """Launches of each kernel that has a row in the profile."""
    lib, ctx = E.b2g_lib(), w.device_context()
    E.b2g_check(lib, ctx, lib.b2g_set_profiling(ctx, 1))
    w.step(steps)
    rows, n = np.zeros(32, PROFILE), ctypes.c_int()
    E.b2g_check(lib, ctx, lib.b2g_get_profile(ctx, E.ptr(rows), 32, ctypes.byref(n)))
    E.b2g_check(lib, ctx, lib.b2g_set_profiling(ctx, 0))
    return {r["name"].decode(): int(r["launches"]) for r in rows}


def test_a_full_set_of_colours_gets_no_team(gpu):
    """A plank under 4100 boxes fills every colour: its thin ones are faster
    fused, so the team solve leaves it alone while a pile of the size gets it."""
    for kind, steps, want in (("plank", 70, 0), ("world", 150, 10)):
        w = gpu.world(kind, 4100, 3, sleep=False)
        w.step(steps)
        assert launches(w, 10)["k_solve_team"] == want, kind
        w.close()


@pytest.mark.parametrize("kind, n, before, want", [
    ("pile", 500, 2, 10), ("pile", 1535, 2, 10), ("pile", 1536, 2, 0), ("pile", 3000, 2, 0), ("pile", 3000, 250, 10),
    ("pendulums", 100, 2, 10), ("pendulums", 383, 2, 10), ("pendulums", 384, 2, 0), ("pendulums", 3000, 2, 0),
    ("chains", 100, 2, 10), ("chains", 400, 2, 0), ("welds", 200, 2, 0), ("wheels", 500, 5, 10), ("wheels", 1300, 5, 0),
])
def test_what_is_a_small_world(gpu, kind, n, before, want):
    """Worlds of many joints, or of many bodies and no contact, are slower in
    one workgroup than stage by stage; either way the steps are the same."""
    a, b = gpu.world(kind, n, 3, sleep=False), gpu.world(kind, n, 3, sleep=False)
    a_launch_per_colour(b)
    a.step(before)
    b.step(before)
    contacts = len(a.contacts()[0])
    assert launches(a, 10)["k_small_prepare"] == want, contacts
    b.step(10)
    same([state(a)], [state(b)])
    a.close(); b.close()


def test_two_worlds_at_once(gpu):
    """Two contexts stepped by two threads, whose teams share the chip."""
    def go(seed, out):
        w = gpu.world("world", 6000, seed, sleep=False)
        out.append(run(w, False, 300))

    alone, both = [], [[], []]
    for seed in (1, 2):
        out = []
        go(seed, out)
        alone.append(out[0])
    threads = [threading.Thread(target=go, args=(seed, both[seed - 1])) for seed in (1, 2)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    for i in range(2):
        same(alone[i], both[i][0])


def test_many_new_pairs_at_once(gpu):
    """A world pressed together: more new pairs than the LDS sort takes, then more contacts than the small-world
    kernels take, then neither."""
    out = []
    for per_colour in (False, True):
        w = gpu.world("world", 1500, 7, sleep=False)
        if per_colour:
            a_launch_per_colour(w)
        w.step(20)
        ctx, lib = w.device_context(), E.b2g_lib()
        bodies = np.zeros(1501, BODY)
        E.b2g_check(lib, ctx, lib.b2g_get_bodies(ctx, 0, 1501, E.ptr(bodies)))
        for k in ("c", "c0"):
            bodies[k][1:] *= np.float32(0.3)
        bodies["xf"][1:, :2] *= np.float32(0.3)
        E.b2g_check(lib, ctx, lib.b2g_set_bodies(ctx, 0, 1501, E.ptr(bodies)))
        states, pairs = [], 0
        for _ in range(4):
            w.step(1)
            states.append(state(w))
            pairs = max(pairs, int(w.stats()["newPairs"]))
        assert pairs > 4096
        states += run(w, False, 90)
        out.append(states)
    same(*out)


@pytest.mark.parametrize("n", [1200, 2500, 3100, 6000])
def test_all_constraints_new_at_once(gpu, n):
    """A pile taken apart and put back: its constraints are all new in one
    step. Sizes for each way of colouring them: in the small world's kernel,
    from the list by one workgroup (5120 at most), and by rounds over the
    table."""
    lib = E.b2g_lib()
    out = []
    for per_colour in (False, True):
        w = gpu.world("world", n, 7, sleep=False)
        if per_colour:
            a_launch_per_colour(w)
        w.step(500)
        ctx = w.device_context()
        here = np.zeros(n + 1, BODY)
        E.b2g_check(lib, ctx, lib.b2g_get_bodies(ctx, 0, n + 1, E.ptr(here)))
        apart = here.copy()
        for k in ("c", "c0", "xf"):
            apart[k][here["type"] == 2, :2] *= np.float32(4.0)
        settled = int(w.stats()["constraints"])
        E.b2g_check(lib, ctx, lib.b2g_set_bodies(ctx, 0, n + 1, E.ptr(apart)))
        w.step(2)
        assert w.stats()["constraints"] < settled // 4
        E.b2g_check(lib, ctx, lib.b2g_set_bodies(ctx, 0, n + 1, E.ptr(here)))
        states, most = [], 0
        for _ in range(4):
            w.step(1)
            states.append(state(w))
            most = max(most, int(w.stats()["constraints"]))
            conflicts, mask = ctypes.c_int(-1), ctypes.c_int(-1)
            E.b2g_check(lib, ctx, lib.b2g_check_colouring(ctx, ctypes.byref(conflicts), ctypes.byref(mask)))
            assert conflicts.value == 0 and mask.value == 0
        assert most > 0.9 * settled
        assert (n < 2000) or (most <= 5120) == (n < 3000)
        w.close()
        out.append(states)
    same(*out)
