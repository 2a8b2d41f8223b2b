"""ymrt_frame_stats counts the kernels that were launched: one per pass for
traversal, and for the stages that fill a queue first one (chunks of up to
65536 paths) or three more; shading takes one for all classes of vertices (up
to 262144 paths) or one for each of its three, with media four."""
import pytest

import ymrt_amd
from ymrt_amd import abi, scenes

pytestmark = pytest.mark.gpu


# paths of the frame (in whole tiles): below, between and above the two bounds
@pytest.mark.parametrize("w,h,spp,fill,classes", [(64, 48, 2, 1, 1), (256, 256, 2, 3, 1), (512, 256, 3, 3, 3)])
@pytest.mark.parametrize("media", [False, True])
def test_launches_are_those_made(gpu_ctx, media, w, h, spp, fill, classes):
    sa = scenes.cornell_media(w, h, grid=False) if media else scenes.cornell_box(w, h)
    sc = ymrt_amd.Scene(gpu_ctx, sa)
    rs = abi.render_settings(w, h, spp, 6, volume=int(media))
    _, st = sc.render_frame(rs, 1, timing=True)
    assert st.chunks == 1 and st.launches_extend == st.launches_shadow == st.passes > 0
    fills = fill * st.passes
    if media:
        assert st.launches_medium == st.launches_transmit == fills + st.passes
    else:
        assert st.launches_medium == st.launches_transmit == 0
    each = 1 if classes == 1 else classes + int(media)
    first = 7  # passes shaded before the host reads how many paths are left
    assert st.passes >= first
    assert fills + each * first + (st.passes - first) <= st.launches_shade <= fills + each * st.passes
    if each == 1 or st.passes == first:
        assert st.launches_shade == fills + each * st.passes
    # untimed frames report none
    assert sc.render_frame(rs, 1)[1].launches_shade == 0
    sc.close()
