"""b2g_get_bodies against what b2g_add_bodies wrote, bit for bit.

The readback gathers a body per lane, stages workgroups of 256 rows in LDS and
sends chunks of 8192 bodies through a ring of four pinned slots: the sizes
here are the edges of those tiles, odd counts (a row is 104 bytes, so an odd
count ends inside a 16-byte word) and ranges that start anywhere.
"""
import ctypes

import numpy as np
import pytest

import engines as E

pytestmark = pytest.mark.gpu

BODY = np.dtype([
    ("type", "<i4"), ("flags", "<i4"), ("xf", "<f4", 4), ("lc", "<f4", 2), ("c0", "<f4", 2), ("a0", "<f4"),
    ("c", "<f4", 2), ("a", "<f4"), ("v", "<f4", 2), ("w", "<f4"), ("force", "<f4", 2), ("torque", "<f4"),
    ("invMass", "<f4"), ("invI", "<f4"), ("linearDamping", "<f4"), ("angularDamping", "<f4"),
    ("gravityScale", "<f4"), ("sleepTime", "<f4"),
])


@pytest.mark.parametrize("n, first, count", [
    (1, 0, 1), (3, 1, 1), (257, 0, 255), (257, 0, 256), (257, 0, 257), (300, 43, 257),
    (8195, 2, 8191), (8195, 2, 8193), (8195, 3, 8192), (33001, 0, 32768), (33001, 1, 32769), (50001, 0, 50001),
])
def test_rows_come_back_as_written(n, first, count):
    lib = E.b2g_lib()
    ctx = E.VP()
    assert lib.b2g_create(ctypes.byref(ctx), 0) == 0
    try:
        rng = np.random.default_rng(n)
        bodies = rng.standard_normal((n, BODY.itemsize // 4)).astype(np.float32).view(BODY)[:, 0]
        bodies["type"] = rng.integers(0, 3, n)
        bodies["flags"] = rng.integers(0, 64, n)
        E.b2g_check(lib, ctx, lib.b2g_add_bodies(ctx, E.ptr(bodies), n, None))
        for _ in range(2):
            out = np.full(count + 1, 7, np.uint8).astype(BODY)
            guard = out[count].tobytes()
            E.b2g_check(lib, ctx, lib.b2g_get_bodies(ctx, first, count, E.ptr(out)))
            assert out[:count].tobytes() == bodies[first:first + count].tobytes()
            assert out[count].tobytes() == guard
    finally:
        lib.b2g_destroy(ctx)
