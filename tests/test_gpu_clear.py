"""Outputs of views with few triangles start from zero in every frame: a frame that covers the view and the shadow map, then
on the same renderer one that leaves most of both empty, at sizes whose words are no multiple of four."""
import numpy as np
import pytest

import oracle
import rosy_amd
from rosy_amd import abi
from scenes import CustomScene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("samples", [1, 4])
@pytest.mark.parametrize("w,h,shadow", [(1, 1, 1), (5, 3, 3), (37, 21, 5), (64, 64, 64), (301, 99, 33)])
def test_second_frame_is_clear(w, h, shadow, samples):
    full = [(-1, -1, 0.5), (3, -1, 0.5), (-1, 3, 0.5)]
    small = [(0.6, 0.6, 0.4), (0.9, 0.6, 0.4), (0.6, 0.9, 0.4)]
    r = rosy_amd.Renderer(device=0)
    try:
        for pos in (full, small):
            sc = CustomScene(pos, [0, 1, 2], w, h, shadow_size=shadow)
            rs = sc.s.raster_state
            rs.msaa_samples = samples
            r.load(sc)
            r.render(sc.frame_desc(abi.SHADE_PLAIN))
            vp, light = sc.camera_views()[0].view_projection[:], sc.cascades()[0].light_view_projection[:]
            want = oracle.raster_view_msaa(sc, vp, w, h, rs) if samples == 4 else oracle.raster_view(sc, vp, w, h, False, rs)[0]
            assert np.array_equal(r.visibility(0), want)
            shadow_want, _ = oracle.raster_view(sc, light, shadow, shadow, True, rs)
            assert np.array_equal(r.shadow_map(0).view(np.uint32), shadow_want.view(np.uint32))
        assert (want == 0).sum() >= want.size // 2
    finally:
        r.close()
