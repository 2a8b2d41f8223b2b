"""Chunks of up to 65536 path slots are compacted by one launch; longer ones, and
many of them in a batch (chunks times the square of the longest above 2^34), by
three.  Up to 262144 paths share one shading launch, longer ones get one per
class.  path_capacity sets the chunk, so the same frame runs through either;
its image must not change, at chunks around a block's 1024 slots, the bound
and odd pixel counts, nor that of a frame of a batch on either side."""
import pytest

import ymrt_amd
from ymrt_amd import abi, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,spp", [(67, 45, 23), (272, 256, 1), (264, 256, 4)])
def test_chunk_sizes_keep_the_frame(gpu_ctx, w, h, spp):
    import torch
    sc = ymrt_amd.Scene(gpu_ctx, scenes.cornell_media(w, h, grid=False))
    ref, _ = sc.render_frame(abi.render_settings(w, h, spp, 4, volume=1), 2)  # more than 65536 slots: three launches
    for cap in (1000, 1024, 1025, 5000, 65535, 65536):
        img, st = sc.render_frame(abi.render_settings(w, h, spp, 4, volume=1, path_capacity=cap), 2)
        assert st.chunks > 1 and torch.equal(img, ref), cap
    sc.close()


@pytest.mark.parametrize("size,counts", [((256, 256), (4, 5)), ((128, 128), (64,)), ((144, 128), (40, 41))])
def test_chunk_counts_keep_the_frames(gpu_ctx, size, counts):
    """Batches whose rounds are compacted by one launch and by three."""
    import torch
    w, h = size
    scene = [ymrt_amd.Scene(gpu_ctx, scenes.cornell_media(w, h, grid=False, halton_seed=s)) for s in range(3)]
    rs = abi.render_settings(w, h, 1, 4, volume=1)
    want = [sc.render_frame(rs, 2)[0] for sc in scene]
    for count in counts:
        jobs = [(scene[i % 3], rs, 2) for i in range(count)]
        for i, (img, _) in enumerate(gpu_ctx.render_batch(jobs)):
            assert torch.equal(img, want[i % 3]), (count, i)
    for sc in scene:
        sc.close()


@pytest.mark.parametrize("w,h,spp", [(45, 31, 2), (331, 257, 4)])
def test_graph_frames_in_one_shading_launch_and_by_class(gpu_ctx, w, h, spp):
    """A frame with texture graphs and no media shades all classes in one launch,
    in rounds shared with a medium it takes one per class."""
    import torch
    graph = ymrt_amd.Scene(gpu_ctx, scenes.textured_box(w, h))
    fog = ymrt_amd.Scene(gpu_ctx, scenes.cornell_media(64, 48, grid=False))
    rs, rf = abi.render_settings(w, h, spp, 5), abi.render_settings(64, 48, 1, 5, volume=1)
    want, st = graph.render_frame(rs, 3, timing=True)
    assert st.launches_shade == (1 if w * h * spp < 65536 else 3) * st.passes + st.passes
    (img, _), (mist, _) = gpu_ctx.render_batch([(graph, rs, 3), (fog, rf, 3)])
    assert torch.equal(img, want) and torch.equal(mist, fog.render_frame(rf, 3)[0])
    graph.close()
    fog.close()
