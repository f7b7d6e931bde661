"""The step's rotations (b2g_sincos_batch) where their evaluation can go wrong.

A double argument reduction and Taylor series serve angles below 2^19 rad, the
device library the others and the values next to a midpoint of two floats.
Both are within a few ulp of a double of the truth, and so is the host's
double sine, so the FP32 roundings agree unless the true value lies within
about 2^-49 of a midpoint: of n values, 2 n * 2^-24 are expected to, at most.
"""
import ctypes

import numpy as np
import pytest

import engines as E

pytestmark = pytest.mark.gpu


def angles(kind):
    g = np.random.default_rng(5)
    if kind == "uniform":
        return g.uniform(-100.0, 100.0, 4_000_000).astype(np.float32)
    if kind == "magnitudes":  # from subnormals to beyond the fast range
        return (np.exp2(g.uniform(-149, 40, 1_000_000)) * g.choice([-1.0, 1.0], 1_000_000)).astype(np.float32)
    if kind == "quadrants":  # floats around multiples of pi / 4
        n = g.integers(-600_000, 600_000, 300_000)
        base = (n * (np.pi / 4)).astype(np.float32)
        return np.concatenate([base, np.nextafter(base, np.float32(np.inf)), np.nextafter(base, np.float32(-np.inf))])
    lim = np.float32(524288.0)
    return np.array([0.0, -0.0, lim, -lim, np.nextafter(lim, np.float32(0)), np.nextafter(lim, np.float32(np.inf)),
                     np.finfo(np.float32).max, np.finfo(np.float32).tiny, 1e-45, -1e-45], np.float32)


@pytest.mark.parametrize("kind", ["uniform", "magnitudes", "quadrants", "special"])
def test_rotation_rounds_the_double(kind):
    a = angles(kind)
    s, c = np.zeros_like(a), np.zeros_like(a)
    lib = E.b2g_lib()
    ctx = E.VP()
    assert lib.b2g_create(ctypes.byref(ctx), 0) == 0
    try:
        E.b2g_check(lib, ctx, lib.b2g_sincos_batch(ctx, E.ptr(a), len(a), E.ptr(s), E.ptr(c)))
    finally:
        lib.b2g_destroy(ctx)
    want_s, want_c = np.sin(a.astype(np.float64)).astype(np.float32), np.cos(a.astype(np.float64)).astype(np.float32)
    for got, want in ((s, want_s), (c, want_c)):
        differ = got.view(np.uint32) != want.view(np.uint32)
        assert differ.sum() <= 2 * len(a) / 2.0 ** 24 + 1
        assert np.all(np.abs(got[differ] - want[differ]) <= np.spacing(np.abs(want[differ])))


def test_rotation_of_nothing_finite():
    a = np.array([np.inf, -np.inf, np.nan], np.float32)
    s, c = np.zeros_like(a), np.zeros_like(a)
    lib = E.b2g_lib()
    ctx = E.VP()
    assert lib.b2g_create(ctypes.byref(ctx), 0) == 0
    try:
        E.b2g_check(lib, ctx, lib.b2g_sincos_batch(ctx, E.ptr(a), len(a), E.ptr(s), E.ptr(c)))
    finally:
        lib.b2g_destroy(ctx)
    assert np.all(np.isnan(s)) and np.all(np.isnan(c))
