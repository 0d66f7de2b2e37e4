"""Paths at the far end of their ranges: as many views as a frame takes, each with a blended pass; mip chains of fourteen
and more levels, built and packed; outputs of megabytes cleared for a view of two triangles."""
import numpy as np
import pytest

import oracle
import rosy_amd
from oracle import textures as tx
from rosy_amd import abi
from scenes import CustomScene
from test_gpu_packed_materials import grid_scene
from test_gpu_textures import read, renderer, upload  # noqa: F401
from test_oracle_shading import scene_data

pytestmark = pytest.mark.gpu


def test_every_view_is_counted():
    scene = rosy_amd.Scene(3, seed=5, total_triangles=20000, width=64, height=48, shadow_size=64, texture_size=16,
                           n_materials=2, n_translucent=2)
    r = rosy_amd.Renderer(device=0)
    try:
        r.load(scene)
        one = scene.frame_desc(abi.SHADE_PLAIN)
        r.render(one)
        image, single = r.color(0), r.stats()
        cams = (abi.CameraView * 15)(*[scene.camera_views()[0]] * 15)
        frame = scene.frame_desc(abi.SHADE_PLAIN)
        frame.n_camera_views, frame.camera_views = 15, cams
        r.render(frame)
        # one cascade and fifteen cameras with their blended lists, 31 views: the cascade is counted once
        r.synchronize()
        many = r.stats()
        shadow = 15 * single.triangles_setup - many.triangles_setup
        assert many.overflowed == 0 and shadow % 14 == 0 and 0 < shadow // 14 < single.triangles_setup
        assert (15 * single.tile_pairs - many.tile_pairs) % 14 == 0 and many.tile_pairs > 14 * single.tile_pairs // 2
        for v in range(15):
            assert np.array_equal(r.color(v), image)
        # an overflow of any of them is seen
        r.set_debug_flags(abi.DEBUG_MIN_CAPACITY)
        r.render(scene.frame_desc(abi.SHADE_NONE))
        r.synchronize()
        r.render(frame)
        assert r.stats().overflowed > 0
        for v in range(15):
            assert np.array_equal(r.color(v), image)
    finally:
        r.close()
        scene.close()


@pytest.mark.parametrize("w,h", [(8192, 3), (3, 9001), (16384, 1), (1, 16384)])
def test_long_chains_are_built(renderer, w, h):  # noqa: F811
    rng = np.random.default_rng(w)
    ups, want = [], []
    for fmt, ch, srgb in ((abi.TEX_RGBA8_SRGB, 4, True), (abi.TEX_RG8_UNORM, 2, False)):
        px = rng.integers(0, 256, (h, w, ch), dtype=np.uint8)
        ups.append((w, h, fmt, abi.MIPS_BUILD, px.tobytes()))
        want.append(tx.mip_chain(px, srgb))
    assert upload(renderer, ups) == abi.RSY_OK
    for t in range(2):
        for l, level in enumerate(want[t]):
            assert np.array_equal(read(renderer, t, l, w, h, level.shape[2]), level), (t, l)


@pytest.mark.parametrize("samples", [1, 4])
def test_long_chains_are_packed(samples):
    sizes = [(8192, 4), (3, 9001), (16384, 2)]
    r = rosy_amd.Renderer(device=0)
    try:
        out = []
        for packed in (True, False):
            sc = grid_scene(sizes, True, packed, samples)
            r.load(sc)
            assert r.packed_materials()[0] == (3 if packed else 0)
            r.update(scene_data(sc, fragment_output=0, light_enabled=0), sc.s.raster_state)
            r.render(sc.frame_desc(abi.SHADE_PLAIN))
            out.append(r.color(0).astype(np.float64))
        assert np.abs(out[0] - out[1]).max() <= 2e-6  # at most ten roundings of 2^-24 on either side
        assert np.unique(out[0][..., 0]).size > 50
    finally:
        r.close()


@pytest.mark.parametrize("samples", [1, 4])
def test_large_outputs_are_cleared(samples):
    w, h, shadow = 2049, 1501, 1999
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
        assert np.array_equal(r.visibility(0), want) and 0 < (want != 0).sum() < want.size // 2
        shadow_want, _ = oracle.raster_view(sc, light, shadow, shadow, True, rs)
        assert np.array_equal(r.shadow_map(0).view(np.uint32), shadow_want.view(np.uint32))
    finally:
        r.close()
