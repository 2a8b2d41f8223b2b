"""The node visit's slab test takes each axis' near plane by the sign of the
ray's reciprocal direction instead of ordering the two products with minimum
and maximum (ymrt_amd/csrc/dev_traverse.hpp visit_node).  Restated in float32
here: both give the same bits for every box with lo <= hi as long as the
reciprocals are finite, an empty child's inverted infinite bounds miss every
such ray, and an infinite reciprocal is what can tell the two apart (so the
kernel sends those lanes through the ordered form)."""
import numpy as np
import pytest

F = np.float32
ROBUST = F(1.0) + F(2.0) * (F(3.0) * F(np.finfo(np.float32).eps) * F(0.5) /
                            (F(1.0) - F(3.0) * F(np.finfo(np.float32).eps) * F(0.5)))


def ordered(lo, hi, o, inv):
    with np.errstate(all="ignore"):
        a, b = (lo - o) * inv, (hi - o) * inv
        return np.fmax.reduce(np.fmin(a, b), axis=-1), np.fmin.reduce(np.fmax(a, b), axis=-1) * ROBUST


def by_sign(lo, hi, o, inv):
    neg = np.signbit(inv)
    with np.errstate(all="ignore"):
        a = (np.where(neg, hi, lo) - o) * inv
        b = (np.where(neg, lo, hi) - o) * inv
        return np.fmax.reduce(a, axis=-1), np.fmin.reduce(b, axis=-1) * ROBUST


def rays(rng, n, kind):
    lo = rng.uniform(-4, 4, (n, 3)).astype(F)
    hi = lo + rng.choice([0.0, 1e-7, 0.3, 5.0], (n, 3)).astype(F)
    hi = np.maximum(lo, hi)
    o = rng.uniform(-6, 6, (n, 3)).astype(F)
    d = rng.normal(size=(n, 3)).astype(F)
    if kind == "on_faces":      # origins in the planes of the box
        pick = rng.integers(0, 3, (n, 3))
        o = np.where(pick == 0, lo, np.where(pick == 1, hi, o))
    elif kind == "tiny":        # reciprocals up to the largest finite ones
        d *= rng.choice([1e-30, 1e-37, 1.0], (n, 3)).astype(F)
    elif kind == "huge":
        o *= F(1e20)
        d *= rng.choice([1e30, 1.0], (n, 3)).astype(F)
    return lo, hi, o, d


@pytest.mark.parametrize("kind", ["plain", "on_faces", "tiny", "huge"])
def test_same_bits_for_finite_reciprocals(kind):
    lo, hi, o, d = rays(np.random.default_rng(5), 200000, kind)
    with np.errstate(all="ignore"):
        inv = F(1.0) / d
    ok = np.isfinite(inv).all(axis=1)
    assert ok.mean() > 0.5
    lo, hi, o, inv = lo[ok], hi[ok], o[ok], inv[ok]
    n0, f0 = ordered(lo, hi, o, inv)
    n1, f1 = by_sign(lo, hi, o, inv)
    # -0 and +0 compare equal, which is all that the test and the sort do
    assert np.array_equal(n0, n1, equal_nan=True) and np.array_equal(f0, f1, equal_nan=True)


@pytest.mark.parametrize("kind", ["plain", "on_faces", "tiny", "huge"])
def test_empty_child_misses(kind):
    _, _, o, d = rays(np.random.default_rng(6), 100000, kind)
    with np.errstate(all="ignore"):
        inv = F(1.0) / d
    ok = np.isfinite(inv).all(axis=1)
    lo, hi = np.full_like(o, np.inf), np.full_like(o, -np.inf)
    tn, tf = by_sign(lo, hi, o, inv)
    assert not ((tf > np.fmax(tn, F(0))) & ok).any()


def test_infinite_reciprocal_needs_the_ordered_form():
    """A ray in the x = lo plane with no x direction: 0 * inf."""
    lo, hi = np.zeros((1, 3), F), np.ones((1, 3), F)
    o, inv = np.array([[0.0, 0.5, -1.0]], F), np.array([[np.inf, np.inf, 1.0]], F)
    n0, f0 = ordered(lo, hi, o, inv)
    n1, f1 = by_sign(lo, hi, o, inv)
    assert not (f0 > n0).any() and (f1 > n1).all()
