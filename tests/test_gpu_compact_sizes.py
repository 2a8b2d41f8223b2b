"""Chunks of up to 65536 path slots are compacted by one launch, longer ones by
three; up to 262144 paths share one shading launch, longer ones get one per
class.  path_capacity sets the chunk, so the same frame runs through either;
its image must not change, at chunks around a block's 1024 slots, the bound
and odd pixel counts."""
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
