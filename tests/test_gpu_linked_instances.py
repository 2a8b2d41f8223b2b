"""Meshes of identity instances are linked into the top-level trees and their
rays never enter an instance; every other instance is entered with a
transformed ray.  A world-to-object x translation of 1e-30 forces the entry
and moves no ray whose x is not tiny, so both ways must give the same bits:
hits with their sides, any-hit flags, visit counts and frames (with media,
whose nearby-instance lists follow the order of instances along a ray)."""
import numpy as np
import pytest

import ymrt_amd
from ymrt_amd import abi, scenes

pytestmark = pytest.mark.gpu


def shared_mesh():
    """One mesh under two identity instances of different materials (the first
    is linked, the second entered: equal distances, the later test wins) and
    a moved one, in a medium box that touches the mesh's bottom face."""
    sa = abi.SceneArrays()
    a = sa.add_material(abi.default_material(diffuse_albedo=(0.8, 0.3, 0.3), specular_weight=0.0))
    glass = sa.add_material(abi.default_material(transmission_weight=1.0, ior_n=1.4, ior_priority=2,
                                                 roughness_x=0.1, roughness_y=0.1))
    m = scenes._add(sa, scenes.box((1.0, 0.5, -1.0), (2.0, 1.5, 0.0)))
    sa.add_instance(m, a)
    sa.add_instance(m, glass)
    sa.add_instance(m, glass, scenes._translate(1.4, 0.25, 0.4))
    sa.add_instance(scenes._add(sa, scenes.quad((-9, 0.5, -9), (-9, 0.5, 9), (9, 0.5, 9), (9, 0.5, -9))), a)
    vol = sa.add_volume((0.4, 0.3, 0.2), (0.9, 0.9, 0.9), 0.1)
    sa.add_instance(scenes._add(sa, scenes.box((0.5, 0.5, -2.0), (4.0, 2.5, 1.5))),
                    sa.add_material(abi.default_material(ior_n=1.0)), inner_volume=vol, boundary=True)
    lq = scenes.quad((1.0, 3.0, -1.0), (2.0, 3.0, -1.0), (2.0, 3.0, 0.0), (1.0, 3.0, 0.0))
    sa.add_instance(scenes._add(sa, lq), sa.add_material(abi.light_material((1.0, 1.0, 1.0), 9.0)))
    sa.set_camera((2.2, 1.4, 4.0), (1.9, 1.0, 0.0), 50.0, 1.0)
    return sa


def entered(sa):
    for it in sa.instances:
        if it["geometry_type"] == abi.GEOMETRY_MESH and np.array_equal(it["w2o"], np.eye(4)):
            w2o = it["w2o"].copy()
            w2o[0, 3] = 1e-30
            it["w2o"] = w2o
    return sa


SCENES = {"shared": shared_mesh, "interior": lambda: scenes.interior(40, 24, tex_size=16),
          "outdoor": lambda: scenes.outdoor(40, 30, fog=True)}


@pytest.mark.parametrize("name", sorted(SCENES))
def test_linked_equals_entered(gpu_ctx, name):
    import torch
    sa, sb = SCENES[name](), entered(SCENES[name]())
    a, b = ymrt_amd.Scene(gpu_ctx, sa), ymrt_amd.Scene(gpu_ctx, sb)
    closest, shadow = scenes.stress_rays(sa, 60001)
    ra, rb = ymrt_amd.Scene.rays_to_device(closest), ymrt_amd.Scene.rays_to_device(shadow)
    ha, va = a.trace_closest(ra, counted=True)
    hb, vb = b.trace_closest(ra, counted=True)
    assert torch.equal(ha, hb) and torch.equal(va, vb)
    assert 0.2 < (ha[:, 2] != -1).float().mean() and (ha[:, 3] != 0).any()
    assert torch.equal(a.trace_any(rb), b.trace_any(rb))
    rs = abi.render_settings(40, 24, 6, 6, volume=1, distant_light=int(name == "outdoor"))
    ia, sta = a.render_frame(rs, 2)
    ib, stb = b.render_frame(rs, 2)
    assert torch.equal(ia, ib)
    assert (sta.extension_rays, sta.extend_nodes, sta.extend_tris, sta.shadow_rays, sta.transmittance_rays) == \
        (stb.extension_rays, stb.extend_nodes, stb.extend_tris, stb.shadow_rays, stb.transmittance_rays)
