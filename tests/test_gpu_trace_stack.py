"""Ray queries keep 16 stack entries per lane in LDS and deeper ones in private
memory when a call has more than one wave per SIMD, and the whole stack in LDS
below that.  The same rays, asked in calls of either size, get the same
answers, with stacks that outgrow the 16 entries."""
import pytest

import ymrt_amd
from ymrt_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side", [65, 400])
def test_large_and_small_calls_agree(gpu_ctx, side):
    import torch
    sa = scenes.heightfield(side)
    sc = ymrt_amd.Scene(gpu_ctx, sa)
    assert sc.info().max_stack > 16
    n = 65536 + 4097  # more than 1024 waves
    closest, shadow = scenes.stress_rays(sa, n)
    # grazing rays along the field cross the most boxes
    closest["d"][::3, 1] *= 0.02
    shadow["d"][::3, 1] *= 0.02
    rc, rs = ymrt_amd.Scene.rays_to_device(closest), ymrt_amd.Scene.rays_to_device(shadow)
    hits, occ = sc.trace_closest(rc), sc.trace_any(rs)
    _, visits = sc.trace_closest(rc, counted=True)
    for a in range(0, n, 30000):
        b = min(a + 30000, n)
        assert torch.equal(sc.trace_closest(rc[a:b].contiguous()), hits[a:b])
        assert torch.equal(sc.trace_any(rs[a:b].contiguous()), occ[a:b])
        assert torch.equal(sc.trace_closest(rc[a:b].contiguous(), counted=True)[1], visits[a:b])
    sc.close()
