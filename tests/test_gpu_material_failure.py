"""rsy_set_materials without the memory for its texels: the call fails, the context renders as one without materials
(its buffers, tables and counts agree), and the next call sets materials as on a new context."""
import numpy as np
import pytest

import rosy_amd
from rosy_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("samples", [1, 4])
def test_upload_that_does_not_fit(samples):
    lib = rosy_amd.lib()
    scene = rosy_amd.Scene(1, seed=3, total_triangles=20000, width=160, height=90, shadow_size=128, texture_size=64,
                           n_materials=4)
    s = scene.s
    s.raster_state.msaa_samples = samples
    frame = scene.frame_desc(abi.SHADE_PLAIN)
    r, bare = rosy_amd.Renderer(device=0), rosy_amd.Renderer(device=0)
    try:
        def shaded(renderer):
            renderer.update(s.scene_data, s.raster_state)
            renderer.render(frame)
            return renderer.color(0)

        r.load(scene)
        first = shaded(r)
        pixels = np.zeros(16384 * 16384, np.uint32)  # never read: the images together need 4 TiB
        huge = (abi.TextureDesc * 4096)(*[abi.TextureDesc(16384, 16384, abi.TEX_RGBA8_SRGB, 1, pixels.ctypes.data)] * 4096)
        assert lib.rsy_set_materials(r.ctx, s.materials, 0, huge, 4096, s.samplers, s.n_samplers) != abi.RSY_OK
        assert b"allocate texels" in lib.rsy_last_error(r.ctx)

        bare.load(scene)
        assert lib.rsy_set_materials(bare.ctx, None, 0, None, 0, None, 0) == abi.RSY_OK
        without = shaded(bare)
        assert np.array_equal(shaded(r), without) and not np.array_equal(first, without)
        r.load(scene)
        assert np.array_equal(shaded(r), first)
    finally:
        r.close()
        bare.close()
        scene.close()
