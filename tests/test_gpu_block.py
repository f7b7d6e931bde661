"""The block solve (one workgroup, bodies in LDS, rows in registers) against a
launch per colour (schedule field tailColours 0), bit for bit.

Sizes around where the path or its layout changes: below and beyond the rows
that lanes hold in registers (1024 with 256 lanes, 2048 with 512; 768 and 1536
with joints), the largest number of bodies in LDS and one beyond it, every
joint type, a body in more contacts than there are colours (the overflow
colour, left to the per-colour kernels), islands that sleep, few iterations.
"""
import numpy as np
import pytest

import engines as E

pytestmark = pytest.mark.gpu


def run(gpu, kind, n, seed, steps, sleep, vel, pos, per_colour):
    w = gpu.world(kind, n, seed, sleep=sleep)
    try:
        if per_colour:
            ctx = w.device_context()
            lib = E.b2g_lib()
            sched = np.zeros(1, E.SCHEDULE)
            E.b2g_check(lib, ctx, lib.b2g_get_schedule(ctx, E.ptr(sched)))
            sched["tailColours"] = 0
            E.b2g_check(lib, ctx, lib.b2g_set_schedule(ctx, E.ptr(sched)))
        out = []
        for _ in range(3):
            w.step(steps // 3, vel=vel, pos=pos)
            meta, man = w.contacts()
            st = w.stats()
            out.append((w.bodies().view(np.uint32), meta, E.manifold_bits(man),
                        [int(st[k]) for k in ("contacts", "constraints", "points", "colours", "positionIterations",
                                              "beginEvents", "endEvents")], float(st["minSeparation"])))
        return out
    finally:
        w.close()


@pytest.mark.parametrize("kind, n, seed, steps, sleep, vel, pos", [
    ("pyramid", 1, 0, 60, True, 8, 3), ("pyramid", 12, 0, 90, True, 8, 3), ("pyramid", 33, 0, 30, False, 8, 3),
    ("world", 64, 1, 240, True, 8, 3), ("world", 500, 2, 240, False, 8, 3), ("world", 1000, 3, 300, False, 6, 2),
    ("world", 1700, 4, 330, False, 8, 3), ("world", 4094, 5, 60, False, 8, 3), ("world", 4095, 5, 420, False, 8, 3),
    ("world", 4096, 5, 60, False, 8, 3), ("world", 300, 6, 240, False, 1, 0), ("world", 300, 6, 60, False, 0, 1),
    ("plank", 100, 0, 120, False, 8, 3), ("terrain", 150, 3, 150, True, 8, 3),
    ("chains", 30, 8, 120, True, 8, 3), ("pendulums", 40, 0, 90, False, 8, 3), ("distance", 20, 0, 60, False, 8, 3),
    ("ropes", 20, 0, 60, False, 8, 3), ("welds", 12, 0, 90, True, 8, 3), ("friction", 16, 0, 60, False, 8, 3),
    ("motor", 12, 0, 60, False, 8, 3), ("pulley", 8, 0, 60, False, 8, 3), ("mouse", 8, 0, 60, False, 8, 3),
    ("prismatic", 12, 0, 60, False, 8, 3), ("wheels", 6, 0, 90, False, 8, 3), ("gears", 4, 0, 60, False, 8, 3),
])
def test_equals_a_launch_per_colour(gpu, kind, n, seed, steps, sleep, vel, pos):
    a = run(gpu, kind, n, seed, steps, sleep, vel, pos, False)
    b = run(gpu, kind, n, seed, steps, sleep, vel, pos, True)
    for (ba, ma, na, sa, la), (bb, mb, nb, sb, lb) in zip(a, b):
        assert np.array_equal(ba, bb)
        assert np.array_equal(ma, mb) and np.array_equal(na, nb)
        assert sa == sb and la == lb
