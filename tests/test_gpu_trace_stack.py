"""Ray queries keep a ray's whole stack in LDS while all waves of the call are
resident that way (stacks of 32 entries: any call; 48, 64 and 96 entries: up to
2816, 2304 and 1536 waves of 64 rays), and in larger calls its top 16 or 32
entries there and the deeper ones in a private array.  Whatever the form, every
kernel (closest hit, counted or not, any hit, with and without spheres, each
stack size) gives the hits and visit counts of the same traversal run on the
host with one plain stack, on rays that outgrow the window."""
import numpy as np
import pytest

import host_traverse
import ymrt_amd
from ymrt_amd import abi, scenes

pytestmark = pytest.mark.gpu


def soup(n, size, levels=1, ratio=1.0):
    """Long random triangles, whose boxes overlap so that rays stack up; in
    levels, each a smaller copy towards the origin, which makes the tree deep."""
    sa = abi.SceneArrays()
    rng = np.random.RandomState(1)
    pos = [(rng.uniform(0, 1, (n, 1, 3)) + rng.normal(size=(n, 3, 3)) * size) * ratio ** k for k in range(levels)]
    pos = np.concatenate(pos).reshape(-1, 3).astype(np.float32)
    sa.add_instance(sa.add_mesh(pos, np.arange(len(pos), dtype=np.uint32).reshape(-1, 3)),
                    sa.add_material(abi.default_material()))
    sa.set_camera((0.5, 0.5, 2.0), (0.5, 0.0, 0.5), 45.0, 1.0)
    return sa


# the kernel's stack entries, rays of a call with the whole stack in LDS, the
# scene, the entries that rays have to outgrow
@pytest.mark.parametrize("entries,line,shape,window", [(32, None, (2000, 0.2), 0),
                                                       (48, 2816 * 64, (100000, 0.5), 32),
                                                       (64, 2304 * 64, (10000, 1.0, 3, 0.3), 32),
                                                       (96, 1536 * 64, (10000, 1.0, 6, 0.3), 32)])
@pytest.mark.parametrize("sphere", [False, True])
def test_both_forms_give_the_host_traversal(gpu_ctx, entries, line, shape, window, sphere):
    import torch
    sa = soup(*shape)
    host = host_traverse.Mesh(sa)
    n = (line or 70000) + 1  # past the line: the first line rays are a call below it
    closest, shadow = scenes.stress_rays(sa, n)
    # half of the rays run towards the nested triangles, and some any-hit rays
    # end beyond them all: boxes are not tested against tmin, so they go
    # through the whole tree along their line
    d = -closest["o"] + np.random.RandomState(3).normal(size=(n, 3)) * 0.05
    closest["d"][::2] = shadow["d"][::2] = d[::2]
    shadow["tmin"][::8], shadow["tmax"][::8] = 1e30, 1e36
    if sphere:  # around the mesh: met by the rays that leave it
        sa.add_instance(sa.add_sphere(50.0), 0)
    sc = ymrt_amd.Scene(gpu_ctx, sa)
    assert {32: 0, 48: 32, 64: 48, 96: 64}[entries] < sc.info().max_stack <= entries
    rc, rs = ymrt_amd.Scene.rays_to_device(closest), ymrt_amd.Scene.rays_to_device(shadow)

    def ask(a, b):
        c, s = rc[a:b].contiguous(), rs[a:b].contiguous()
        hits, visits = sc.trace_closest(c, counted=True)
        assert torch.equal(sc.trace_closest(c), hits)
        return hits, visits, sc.trace_any(s)

    all_rays = ask(0, n)
    for got, below in zip(all_rays, ask(0, line or n)):
        assert torch.equal(got[:len(below)], below)
    if not sphere:  # the host has the mesh alone: some rays of the call
        m = 6000
        for rays, any_hit, got in ((closest, False, all_rays[0]), (shadow, True, all_rays[2])):
            want, visits, deepest = host.trace(rays[:m], any=any_hit)
            assert deepest > window
            assert np.array_equal(got[:m].cpu().numpy().view(np.uint32), want)
            if not any_hit:
                assert np.array_equal(all_rays[1][:m].cpu().numpy().view(np.uint32), visits)
    else:
        assert ((all_rays[0][:, 2] != -1) & (all_rays[0][:, 1] == -1)).any()  # sphere hits
    sc.close()
