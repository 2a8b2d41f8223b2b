"""The window form of the traversal stack (a ring of 16 entries, deeper ones
apart, the ray setup parked) against the plain stack, on the host: the same
hits, flags and visit counts on rays that hold up to 60 entries."""
import numpy as np
import pytest

import host_traverse
from ymrt_amd import scenes
from test_gpu_trace_stack import soup


@pytest.mark.parametrize("shape", [(2000, 0.2), (3000, 1.0, 6, 0.3)])
def test_window_equals_the_plain_stack(shape):
    sa = soup(*shape)
    mesh = host_traverse.Mesh(sa)
    closest, shadow = scenes.stress_rays(sa, 3000)
    d = -closest["o"] + np.random.RandomState(3).normal(size=closest["o"].shape) * 0.05
    closest["d"][::2] = shadow["d"][::2] = d[::2]
    shadow["tmin"][::8], shadow["tmax"][::8] = 1e30, 1e36
    for rays, any_hit in ((closest, False), (shadow, True)):
        plain, ring = (mesh.trace(rays, any=any_hit, ring=r) for r in (False, True))
        assert plain[2] == ring[2] > 16
        assert np.array_equal(plain[0], ring[0]) and np.array_equal(plain[1], ring[1])
