"""Materials sampled as one packed image against the same maps sampled one by one, for every size, addressing mode
and metallic-roughness form that is packed, magnified and minified, single-level and with mip chains.  The second scene is
the first with one thing changed that no sample depends on but that keeps its materials from being packed: the
normal maps' minification filter (single-level images have no use for it), or their last mip level (never reached)."""
import numpy as np
import pytest

import rosy_amd
from oracle import textures as tx
from rosy_amd import abi
from scenes import CustomScene
from test_oracle_shading import scene_data

pytestmark = pytest.mark.gpu

WRAPS = [(2, 2), (0, 0), (1, 1), (0, 1), (2, 0)]
SINGLE = [(1, 1), (2, 3), (4, 4), (5, 4), (3, 9), (8, 16), (33, 17), (64, 64), (37, 20)]
CHAINS = [(64, 64), (37, 20), (65, 33), (16, 128), (100, 61)]
MR = [(abi.TEX_RG8_SRGB, 2, True), (abi.TEX_RG8_UNORM, 2, False), (abi.TEX_RGBA8_SRGB, 4, True), (abi.TEX_RGBA8_UNORM, 4, False)]


def grid_scene(sizes, chains, packed, samples):
    """One quad of about 48 pixels per size, its addressing, metallic-roughness form and uv span taken in turn."""
    rng = np.random.default_rng(21)
    pos, uvs, tris, draws, textures, materials, samplers = [], [], [], [], [], [], []
    for k, (w, h) in enumerate(sizes):
        cx, cy = k % 3, k // 3
        x0, x1 = -1 + cx * 2 / 3 + 0.031, -1 + (cx + 1) * 2 / 3 - 0.027
        y0, y1 = -1 + cy * 2 / 3 + 0.029, -1 + (cy + 1) * 2 / 3 - 0.033
        u0, u1 = [(-1.3, 2.2), (0.1, 0.6), (-0.2, 1.1)][(k + len(sizes)) % 3]
        base = len(pos)
        pos += [(x0, y0, 0.5), (x1, y0, 0.5), (x1, y1, 0.5), (x0, y1, 0.5)]
        uvs += [(u0, u0), (u1, u0), (u1, u1), (u0, u1)]
        draws.append((len(tris) // 3, 2))
        tris += [base, base + 1, base + 2, base, base + 2, base + 3]
        fmt, ch, srgb = MR[k % 4]
        for f, c, s, lo, hi in ((abi.TEX_RGBA8_SRGB, 4, True, 0, 256), (abi.TEX_RG8_UNORM, 2, False, 64, 193),
                                (fmt, ch, srgb, 0, 256)):
            px = rng.integers(lo, hi, size=(h, w, c), dtype=np.uint8)
            levels = tx.mip_chain(px, s) if chains else [px]
            if chains and not packed and f == abi.TEX_RG8_UNORM and c == 2 and lo == 64:
                levels = levels[:-1]
            textures.append((w, h, f, b"".join(np.ascontiguousarray(x).tobytes() for x in levels), len(levels)))
        ws, wt = WRAPS[k % len(WRAPS)]
        samplers += [(5, 4, ws, wt), (5 if chains or packed else 0, 4, ws, wt)]
        mr = {"mixmap_sampled_image_index": 3 * k + 2, "mixmap_sampler_index": 2 * k} if k % 2 else \
             {"metallic_sampled_image_index": 3 * k + 2, "metallic_sampler_index": 2 * k}
        materials.append({"color_sampled_image_index": 3 * k, "color_sampler_index": 2 * k,
                          "normal_sampled_image_index": 3 * k + 1, "normal_sampler_index": 2 * k + 1, **mr})
    sc = CustomScene(pos, tris, 150, 150, draws=draws, uvs=uvs, textures=textures, materials=materials,
                     material_of_draw=list(range(len(sizes))), samplers=samplers)
    sc.s.scene_data.shadows_enabled = 0
    sc.s.raster_state.msaa_samples = samples
    return sc


@pytest.mark.parametrize("samples", [1, 4])
@pytest.mark.parametrize("sizes,chains", [(SINGLE, False), (CHAINS, True)], ids=["single", "chains"])
def test_packed_equals_one_by_one(sizes, chains, samples):
    r = rosy_amd.Renderer(device=0)
    try:
        out = []
        for packed in (True, False):
            sc = grid_scene(sizes, chains, packed, samples)
            r.load(sc)
            frames = []
            for mode in (0, 13, 14, 15, 6):
                r.update(scene_data(sc, fragment_output=mode, light_enabled=0), sc.s.raster_state)
                r.render(sc.frame_desc(abi.SHADE_PLAIN))
                frames.append(r.color(0).astype(np.float64))
            out.append(frames)
        for mode, a, b in zip((0, 13, 14, 15, 6), *out):
            # sampled values: at most ten roundings of 2^-24 on either side; normals: twice that, bent by at most
            # |m| <= 1 and z >= 0.7, then normalised
            tolerance = 2e-5 if mode == 6 else 2e-6
            assert np.abs(a - b).max() <= tolerance, (mode, np.argwhere(np.abs(a - b) > tolerance)[:4])
            assert np.unique(a[..., 0]).size > 50
    finally:
        r.close()
