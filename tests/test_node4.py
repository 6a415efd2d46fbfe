"""The four-wide node test (planes picked by the ray's signs, infinite boxes for
empty children, slab() itself for rays that may meet a NaN) against slab() on
the boxes as given: same hits, same keys bit for bit. CPU build of the device
code."""
import ctypes as C

import numpy as np
import pytest

import hostpath


def run(lo, hi, count, o, d, best):
    n = o.shape[0]
    f = lambda a: np.ascontiguousarray(a, np.float32).ctypes.data_as(C.POINTER(C.c_float))  # noqa: E731
    c = np.ascontiguousarray(count, np.int32)
    keep = [np.ascontiguousarray(a, np.float32) for a in (lo, hi, o, d, best)]
    differ, hits, odds = C.c_int(0), C.c_int(0), C.c_int(0)
    hostpath.lib().host_node4(n, f(keep[0]), f(keep[1]), c.ctypes.data_as(C.POINTER(C.c_int)), f(keep[2]), f(keep[3]),
                              f(keep[4]), C.byref(differ), C.byref(hits), C.byref(odds))
    return differ.value, hits.value, odds.value


def boxes(rng, n):
    a, b = rng.uniform(-2, 2, (n, 4, 3)), rng.uniform(-2, 2, (n, 4, 3))
    flat = rng.random((n, 4, 3)) < 0.15  # flat boxes
    b = np.where(flat, a, b)
    return np.minimum(a, b).astype(np.float32), np.maximum(a, b).astype(np.float32)


def test_ordinary_rays():
    rng = np.random.default_rng(1)
    n = 200000
    lo, hi = boxes(rng, n)
    o = rng.uniform(-3, 3, (n, 3))
    d = rng.normal(size=(n, 3))
    best = np.where(rng.random(n) < 0.5, 1e6, rng.uniform(0, 3, n))
    differ, hits, odds = run(lo, hi, rng.integers(1, 5, n), o, d, best)
    print(f"{hits} hits of {4 * n} children")
    assert differ == 0 and hits > n // 20 and odds == 0


@pytest.mark.parametrize("seed", range(4))
def test_special_values(seed):
    """Zero, tiny, huge, infinite and NaN directions and origins, origins on
    box planes, boxes with NaN, infinite or swapped planes."""
    rng = np.random.default_rng(10 + seed)
    n = 100000
    lo, hi = boxes(rng, n)
    lo, hi = np.round(lo * 2) / 2, np.round(hi * 2) / 2  # grid-aligned planes
    o = np.round(rng.uniform(-3, 3, (n, 3)) * 2) / 2
    d = np.round(rng.normal(size=(n, 3)))
    vals = np.array([0.0, -0.0, 1.0, -1.0, 1e-30, -1e-30, 1e-42, 1e30, -1e30, np.inf, -np.inf, np.nan], np.float32)

    def sprinkle(a, p):
        m = rng.random(a.shape) < p
        return np.where(m, rng.choice(vals, a.shape), a)

    d = sprinkle(d, 0.3)
    if seed & 1:
        o = sprinkle(o, 0.1)
    if seed & 2:
        lo, hi = sprinkle(lo, 0.03), sprinkle(hi, 0.03)
    best = rng.choice(np.array([1e6, 0.0, 0.5, 2.0, np.inf, -1.0], np.float32), n)
    differ, hits, odds = run(lo, hi, rng.integers(1, 5, n), o, d, best)
    print(f"seed {seed}: {hits} hits, {odds} rays through slab() itself")
    assert differ == 0 and hits > 0 and odds > n // 4
