"""Rays with zero, signed-zero and denormal direction components, origins in
vertex planes (the faces of nodes and boxes, where the slab test meets 0 * inf),
odd intervals, and rays with infinities and NaN: the GPU's hits, any-hit flags
and visit counts are those of the same traversal on the host, bit for bit, on a
mesh that is linked into the top-level tree and on one that rays enter through
a transform.  (test_slab_signs compares the host's node visit with the ordered
slab test on such rays.)"""
import numpy as np
import pytest

import host_traverse
import ymrt_amd
from ymrt_amd import abi, scenes

pytestmark = pytest.mark.gpu


def rays_at(sa, n, rng):
    it, = sa.instances
    pos = sa.meshes[it["mesh"]]["pos"] @ it["o2w"][:3, :3].T + it["o2w"][:3, 3]
    v = pos[rng.integers(0, len(pos), n)].astype(np.float32)
    i = np.arange(n)
    d = np.zeros((n, 3), np.float32)
    axis, sign = rng.integers(0, 3, n), rng.choice([-1.0, 1.0], n)
    d[i, axis] = sign
    two = rng.random(n) < 0.4
    other = (axis + rng.integers(1, 3, n)) % 3
    d[i[two], other[two]] = rng.normal(size=two.sum())
    tiny = rng.random(n) < 0.1
    d[i[tiny], other[tiny]] = rng.choice([1e-38, -1e-41, 1e-45], tiny.sum())
    d = np.where((d == 0) & (rng.random((n, 3)) < 0.5), np.float32(-0.0), d)
    o = v.copy()
    o[i, axis] = v[i, axis] - sign * rng.uniform(0, 2, n)
    shift = rng.random(n) < 0.3
    o[shift] += rng.uniform(-0.3, 0.3, (shift.sum(), 3)).astype(np.float32)
    odd = rng.random(n) < 0.05
    values = np.array([np.inf, -np.inf, np.nan], np.float32)
    d[i[odd], other[odd]] = rng.choice(values, odd.sum())
    odd = rng.random(n) < 0.03
    o[i[odd], axis[odd]] = rng.choice(values, odd.sum())
    r = np.zeros(n, abi.RAY_DTYPE)
    r["o"], r["d"] = o, d
    r["tmin"] = rng.choice([1e-7, 0.0, -1.0], n)
    r["tmax"] = rng.choice([1e36, 1e36, 1.0, 0.0, -0.5], n)
    return r


@pytest.mark.parametrize("entered", [False, True])
def test_axis_rays_equal_the_host_traversal(gpu_ctx, entered):
    sa = scenes.heightfield(65)
    if entered:  # axes swapped and moved: zero components stay zero
        o2w = np.array([[0, 0, 1, 0.25], [1, 0, 0, -0.5], [0, 1, 0, 0.125], [0, 0, 0, 1]], np.float32)
        sa.instances[0]["o2w"] = o2w
        w2o = np.linalg.inv(o2w.astype(np.float64)).astype(np.float32)
        w2o[3] = (0, 0, 0, 1)
        sa.instances[0]["w2o"] = w2o
    rays = rays_at(sa, 200000, np.random.default_rng(3))
    host = host_traverse.Mesh(sa)
    sc = ymrt_amd.Scene(gpu_ctx, sa)
    r = ymrt_amd.Scene.rays_to_device(rays)
    hits, visits = sc.trace_closest(r, counted=True)
    want, want_visits, _ = host.trace(rays)
    got = hits.cpu().numpy().view(np.uint32)
    # a NaN distance has no particular bits
    for h in (got, want):
        h[np.isnan(h[:, 0].copy().view(np.float32)), 0] = 0x7FC00000
    assert np.array_equal(got, want)
    assert np.array_equal(visits.cpu().numpy().view(np.uint32), want_visits)
    assert 0.02 < (want[:, 2] == 0).mean() < 0.9
    occ = sc.trace_any(r).cpu().numpy().view(np.uint32)
    assert np.array_equal(occ, host.trace(rays, any=True)[0])
    sc.close()
