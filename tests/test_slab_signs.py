"""The node visit takes each axis' near plane by the sign of the ray's
reciprocal direction, sends rays with an infinite reciprocal through the
ordered form, and lets an empty child miss by its inverted infinite bounds
(ymrt_amd/csrc/dev_traverse.hpp visit_node).  The visit itself, compiled for
the host, goes on to the children that the ordered form (both products of
every axis through minimum and maximum, empty children left out by their code)
finds, nearest first: for every kind of ray, with the ray's setup fresh and
read back from its parked form."""
import numpy as np
import pytest

import host_traverse
from ymrt_amd import abi

F = np.float32
EMPTY = 0xFFFFFFFF
ROBUST = F(1.0) + F(2.0) * (F(3.0) * F(np.finfo(np.float32).eps) * F(0.5) /
                            (F(1.0) - F(3.0) * F(np.finfo(np.float32).eps) * F(0.5)))


def ordered(lo, hi, child, rays):
    """Distances of the children hit (n, 4), infinity for the others."""
    with np.errstate(all="ignore"):
        inv = (F(1.0) / rays["d"])[:, None]
        a, b = (lo - rays["o"][:, None]) * inv, (hi - rays["o"][:, None]) * inv
        tn = np.fmax.reduce(np.fmin(a, b), axis=-1)
        tf = np.fmin.reduce(np.fmax(a, b), axis=-1) * ROBUST
        hit = (child != EMPTY) & (tf > tn) & (tf > 0) & (tn <= rays["tmax"][:, None])
    return np.where(hit, np.maximum(tn, F(0.0)), F(np.inf))


def cases(rng, n, kind):
    lo = rng.uniform(-4, 4, (n, 4, 3)).astype(F)
    hi = lo + rng.choice([0.0, 1e-7, 1.0, 8.0, 8.0], (n, 4, 3)).astype(F)
    child = np.where(rng.random((n, 4)) < 0.25, EMPTY, np.arange(4 * n).reshape(n, 4))
    rays = np.zeros(n, abi.RAY_DTYPE)
    o = rng.uniform(-6, 6, (n, 3)).astype(F)
    # half of the rays run at a point of a child's box
    at = rng.integers(0, 4, n)
    p = lo[np.arange(n), at] + rng.random((n, 3)) * (hi - lo)[np.arange(n), at]
    if kind in ("on_faces", "zeros_on_faces"):
        pick = rng.integers(0, 6, (n, 3))
        o = np.where(pick == 0, lo[np.arange(n), at], np.where(pick == 1, hi[np.arange(n), at], o))
    d = np.where(rng.random((n, 1)) < 0.5, p - o, rng.normal(size=(n, 3))).astype(F)
    if kind in ("zeros", "zeros_on_faces"):
        d = np.where(rng.random((n, 3)) < 0.5, np.where(rng.random((n, 3)) < 0.5, F(0.0), F(-0.0)), d)
    elif kind == "tiny":        # reciprocals up to the largest finite ones, and past them
        d *= rng.choice([1e-30, 1e-37, 1e-42, 1.0], (n, 3)).astype(F)
    elif kind == "huge":
        o *= rng.choice([1e20, 1.0, 1.0, 1.0], (n, 1)).astype(F)
        d *= rng.choice([1e30, 1.0], (n, 1)).astype(F)
    elif kind == "not_finite":
        odd = np.array([np.inf, -np.inf, np.nan], F)
        d = np.where(rng.random((n, 3)) < 0.3, rng.choice(odd, (n, 3)), d)
        o = np.where(rng.random((n, 3)) < 0.2, rng.choice(odd, (n, 3)), o)
    rays["o"], rays["d"] = o, d
    rays["tmax"] = rng.choice(np.array([1e36, 1e36, 1e36, 1e36, 3.0, 0.0, -0.5], F), n)
    lo[child == EMPTY], hi[child == EMPTY] = np.inf, -np.inf
    return lo, hi, child, rays


@pytest.mark.parametrize("park", [False, True])
@pytest.mark.parametrize("kind", ["plain", "on_faces", "zeros", "zeros_on_faces", "tiny", "huge", "not_finite"])
def test_visit_follows_the_ordered_form(kind, park):
    n = 100000
    lo, hi, child, rays = cases(np.random.default_rng(5), n, kind)
    want = ordered(lo, hi, child, rays)
    hit = np.isfinite(want)
    assert hit.sum() > 5000 and (~hit & (child != EMPTY)).sum() > 5000
    got = host_traverse.visit(host_traverse.nodes(lo, hi, child), rays, park)
    # which children: the same ones, each once
    row = np.arange(n)[:, None]
    went = np.zeros((n, 4), bool)
    live = got != EMPTY
    assert (got[live] // 4 == np.broadcast_to(row, got.shape)[live]).all()
    went[np.broadcast_to(row, got.shape)[live], got[live] % 4] = True
    assert np.array_equal(went, hit) and live.sum() == went.sum()
    # in what order: nearest first (equal distances in either)
    dist = np.where(live, want[row, got % 4], F(np.inf))
    assert (dist[:, 1:] >= dist[:, :-1]).all()


def test_infinite_reciprocal_needs_the_ordered_form():
    """A ray in the x = lo plane with no x direction: 0 * inf, which the
    ordered form takes for a miss and the planes by sign for a hit."""
    lo, hi = np.zeros((1, 4, 3), F), np.ones((1, 4, 3), F)
    rays = np.zeros(1, abi.RAY_DTYPE)
    rays["o"], rays["d"], rays["tmax"] = (0.0, 0.5, -1.0), (0.0, 0.0, 1.0), 1e36
    child = np.arange(4)[None]
    assert not np.isfinite(ordered(lo, hi, child, rays)).any()
    assert (host_traverse.visit(host_traverse.nodes(lo, hi, child), rays, False) == EMPTY).all()
    with np.errstate(all="ignore"):
        inv = F(1.0) / rays["d"][0]
        near, far = (lo[0, 0] - rays["o"][0]) * inv, (hi[0, 0] - rays["o"][0]) * inv
    assert np.fmin.reduce(far) > max(np.fmax.reduce(near), 0)
