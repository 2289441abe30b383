"""The arithmetic of the three-part bf16 split (vedic_split.hpp), on the CPU:
the parts of a scaled binary32 value sum to it exactly and are zero or normal
over [2^-149, 2^103), values that round to 2^104 or more show, their sizes, and the bound of the product terms that the
six-product form drops."""
import numpy as np
import pytest

SCALE = np.float32(2.0 ** 24)


def bf16(x):
    """binary32 -> bf16 (round to nearest even), as binary32."""
    u = np.asarray(x, np.float32).view(np.uint32).astype(np.uint64)
    u = (u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000
    return u.astype(np.uint32).view(np.float32)


def split(x):
    p1 = bf16(x)
    r = x - p1
    p2 = bf16(r)
    return p1, p2, bf16(r - p2)


def values(lo, hi, n, rng):
    """Binary32 values of random sign, exponent in [lo, hi) and significand."""
    bits = rng.integers(0, 2 ** 23, n, dtype=np.int64)
    v = np.ldexp(1.0 + bits * 2.0 ** -23, rng.integers(lo, hi, n))
    return (np.where(rng.random(n) < 0.5, v, -v)).astype(np.float32)


@pytest.mark.parametrize("lo,hi", [(-149, -126), (-127, -100), (-100, 0), (0, 80), (80, 103)])
def test_parts_are_exact(lo, hi):
    rng = np.random.default_rng(hi - lo)
    x = values(lo, hi, 1 << 18, rng)
    with np.errstate(over="raise"):
        s = x * SCALE
        p = split(s)
    assert np.array_equal(s.astype(np.float64), x.astype(np.float64) * 2.0 ** 24)
    assert np.array_equal(sum(q.astype(np.float64) for q in p), s.astype(np.float64))
    for q in p:
        assert np.all((q == 0) | (np.abs(q) >= np.float32(2.0 ** -126)))
    assert np.all(np.abs(p[1].astype(np.float64)) <= 2.0 ** -8 * np.abs(s))
    assert np.all(np.abs(p[2].astype(np.float64)) <= 2.0 ** -17 * np.abs(s))


@pytest.mark.parametrize("x", [2.0 ** 104, -(2.0 ** 104) * (1 - 2.0 ** -9), 3.4e38, np.inf, -np.inf, np.nan])
def test_past_the_range(x):
    with np.errstate(over="ignore", invalid="ignore"):
        s = np.array([x], np.float32) * SCALE
        assert not all(np.isfinite(q).all() for q in split(s))
    below = np.array([2.0 ** 104 * (1 - 2.0 ** -8)], np.float32) * SCALE
    assert all(np.isfinite(q).all() for q in split(below))


def dropped(x, y):
    a, b = (([q.astype(np.float64) for q in split(v)]) for v in (x, y))
    return np.abs(a[1] * b[2] + a[2] * b[1] + a[2] * b[2]) / np.abs(x.astype(np.float64) * y)


def test_dropped_terms():
    rng = np.random.default_rng(3)
    r = dropped(values(0, 1, 1 << 20, rng), values(0, 1, 1 << 20, rng))
    assert r.max() <= 2.0 ** -24 * (1 + 2.0 ** -10)
    x = np.array([1 + 2.0 ** -8 - 2.0 ** -17], np.float32)
    assert 0.98 * 2.0 ** -24 < dropped(x, x)[0] <= 2.0 ** -24
