"""How the pass kernels deal their queues over the waves of a launch: shares
of 64 to 256 items by queue length, the first of them without atomics, and in
a batch one deal over the queues of all frames.  Whatever the deal, every path
is handled once: frames are bit-identical to the one that a single wave per
kernel renders, which takes every share in order."""
import pytest

import ymrt_amd
from ymrt_amd import abi, scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return ymrt_amd.Context(0)


# paths: below one wave, a ragged few waves, shares between the bounds, and a
# queue long enough for full shares on few waves
@pytest.mark.parametrize("w,h,spp", [(1, 1, 1), (17, 5, 1), (33, 31, 3), (70, 41, 16)])
@pytest.mark.parametrize("scene", ["cornell", "media"])
def test_any_wave_count_gives_the_same_frame(ctx, scene, w, h, spp):
    import torch
    sa = scenes.cornell_box(w, h) if scene == "cornell" else scenes.cornell_media(w, h, grid=True)
    sc = ymrt_amd.Scene(ctx, sa)
    vol = int(scene == "media")
    ref, st = sc.render_frame(abi.render_settings(w, h, spp, 5, volume=vol, persistent_waves=1), 3)
    for waves in (0, 2, 7, 63, 1000):
        img, s2 = sc.render_frame(abi.render_settings(w, h, spp, 5, volume=vol, persistent_waves=waves), 3)
        assert torch.equal(img, ref), waves
        assert (s2.extension_rays, s2.shadow_rays, s2.transmittance_rays) == \
            (st.extension_rays, st.shadow_rays, st.transmittance_rays)
    sc.close()


def test_batch_of_unlike_queues(ctx):
    """One launch over a frame of one pixel, frames of some waves and one that
    holds most of the items: home waves, slots without any, and helpers."""
    import torch
    sizes = [(1, 1, 1), (160, 120, 16), (17, 5, 2), (48, 48, 4), (3, 2, 1), (64, 33, 1)]
    jobs = []
    for i, (w, h, spp) in enumerate(sizes):
        jobs.append((ymrt_amd.Scene(ctx, scenes.cornell_box(w, h, halton_seed=i)),
                     abi.render_settings(w, h, spp, 4), 2))
    for slots in (0, 2, 3):
        for (sc, rs, fr), (img, _) in zip(jobs, ctx.render_batch(jobs, max_slots=slots)):
            assert torch.equal(img, sc.render_frame(rs, fr)[0]), (rs.width, rs.height, slots)
