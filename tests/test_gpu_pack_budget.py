"""Packed copies of materials within their memory: materials that combine the same maps share or repeat copies, up to
twice the texels' memory; a limit that only some materials fit under packs those and samples the others map by map,
to the same image; an upload without packable materials holds no copy."""
import numpy as np
import pytest

import rosy_amd
from oracle import textures as tx
from rosy_amd import abi
from scenes import CustomScene
from test_gpu_neural_eval import images as decoder_images
from test_gpu_packed_materials import CHAINS, SINGLE, WRAPS, grid_scene
from test_oracle_shading import scene_data

pytestmark = pytest.mark.gpu


def tiles(w, h, levels):
    return sum(-(-max(1, w >> l) // 4) * -(-max(1, h >> l) // 4) for l in range(levels))


@pytest.mark.parametrize("sizes,chains", [(SINGLE, False), (CHAINS, True)], ids=["single", "chains"])
def test_every_some_and_no_material_packed(sizes, chains):
    r = rosy_amd.Renderer(device=0)
    try:
        out, used = [], []
        for packed, limited in ((True, False), (True, True), (False, False)):
            r.set_debug_flags(abi.DEBUG_MIN_PACK if limited else 0)
            sc = grid_scene(sizes, chains, packed, 1)
            r.load(sc)
            used.append(r.packed_materials())
            r.update(scene_data(sc, fragment_output=0, light_enabled=0), sc.s.raster_state)
            r.render(sc.frame_desc(abi.SHADE_PLAIN))
            out.append(r.color(0).astype(np.float64))
        size = [128 * tiles(w, h, len(tx.mip_chain(np.zeros((h, w, 4), np.uint8), True)) if chains else 1) for w, h in sizes]
        fit = 0
        n = 0
        for b in size:  # in the materials' order, while they fit
            if fit + b <= 16384:
                fit, n = fit + b, n + 1
        assert used[0] == (len(sizes), sum(size)) and used[1] == (n, fit) and used[2] == (0, 0)
        assert 0 < n < len(sizes)
        # sampled values: at most ten roundings of 2^-24 on either side
        assert np.abs(out[0] - out[1]).max() <= 2e-6 and np.abs(out[0] - out[2]).max() <= 2e-6
    finally:
        r.close()


def test_shared_maps_take_at_most_twice_the_texels():
    rng = np.random.default_rng(4)
    n, w = 12, 32  # n^2 materials from n albedo and n normal maps and one metallic-roughness map
    images = [(abi.TEX_RGBA8_SRGB, 4)] * n + [(abi.TEX_RG8_UNORM, 2)] * n + [(abi.TEX_RG8_UNORM, 2)]
    pixels = [rng.integers(0, 256, (w, w, c), dtype=np.uint8) for _, c in images]
    descs = (abi.TextureDesc * len(images))(*[abi.TextureDesc(w, w, f, 1, p.ctypes.data) for (f, _), p in zip(images, pixels)])
    mats = (abi.GpuMaterial * (n * n))()
    for k in range(n * n):
        for f, _ in abi.GpuMaterial._fields_:
            if f.endswith("_index"):
                setattr(mats[k], f, 0xFFFFFFFF)
        mats[k].color_sampled_image_index = k % n
        mats[k].normal_sampled_image_index = n + k // n
        mats[k].metallic_sampled_image_index = 2 * n
    pool = sum(p.size for p in pixels)  # (multiples of the 256-byte alignment)
    each = w * w * 8
    r = rosy_amd.Renderer(device=0)
    try:
        assert rosy_amd.lib().rsy_set_materials(r.ctx, mats, n * n, descs, len(images), None, 0) == abi.RSY_OK
        count, used = r.packed_materials()
        assert used == count * each and count == 2 * pool // each < n * n
        # each material's maps once: all of them
        assert rosy_amd.lib().rsy_set_materials(r.ctx, mats, n, descs, len(images), None, 0) == abi.RSY_OK
        assert r.packed_materials() == (n, n * each)
        # the same maps under several samplers share one image
        for k in range(n):
            mats[k].color_sampled_image_index = 0
        samplers = (abi.Sampler * 3)(abi.Sampler(4, 4, 0, 0), abi.Sampler(4, 4, 1, 2), abi.Sampler(4, 4, 2, 2))
        for k in range(n):
            mats[k].color_sampler_index = mats[k].normal_sampler_index = mats[k].metallic_sampler_index = k % 3
        assert rosy_amd.lib().rsy_set_materials(r.ctx, mats, n, descs, len(images), samplers, 3) == abi.RSY_OK
        assert r.packed_materials() == (n, each)
    finally:
        r.close()


def shared_scene(packed):
    """One set of maps under every addressing mode, a quad each."""
    rng = np.random.default_rng(8)
    pos, uvs, tris, draws, materials, samplers = [], [], [], [], [], []
    for k, (ws, wt) in enumerate(WRAPS):
        x0, x1 = -1 + 0.4 * k + 0.011, -1 + 0.4 * (k + 1) - 0.013
        base = len(pos)
        pos += [(x0, -0.9, 0.5), (x1, -0.9, 0.5), (x1, 0.9, 0.5), (x0, 0.9, 0.5)]
        uvs += [(-1.3, -1.2), (2.2, -1.2), (2.2, 1.9), (-1.3, 1.9)]
        draws.append((len(tris) // 3, 2))
        tris += [base, base + 1, base + 2, base, base + 2, base + 3]
        samplers += [(5, 4, ws, wt), (5 if packed else 0, 4, ws, wt)]  # (single-level images are never minified)
        materials.append({"color_sampled_image_index": 0, "color_sampler_index": 2 * k, "normal_sampled_image_index": 1,
                          "normal_sampler_index": 2 * k + 1, "metallic_sampled_image_index": 2, "metallic_sampler_index": 2 * k})
    textures = [(13, 10, f, rng.integers(lo, hi, (10, 13, c), dtype=np.uint8).tobytes(), 1)
                for f, c, lo, hi in ((abi.TEX_RGBA8_SRGB, 4, 0, 256), (abi.TEX_RG8_UNORM, 2, 64, 193), (abi.TEX_RG8_UNORM, 2, 0, 256))]
    sc = CustomScene(pos, tris, 150, 40, draws=draws, uvs=uvs, textures=textures, materials=materials,
                     material_of_draw=list(range(len(WRAPS))), samplers=samplers)
    sc.s.scene_data.shadows_enabled = 0
    return sc


def test_one_image_under_several_samplers():
    r = rosy_amd.Renderer(device=0)
    try:
        out = []
        for packed in (True, False):
            sc = shared_scene(packed)
            r.load(sc)
            assert r.packed_materials() == ((len(WRAPS), 128 * tiles(13, 10, 1)) if packed else (0, 0))
            frames = []
            for mode in (0, 13, 14, 15):
                r.update(scene_data(sc, fragment_output=mode, light_enabled=0), sc.s.raster_state)
                r.render(sc.frame_desc(abi.SHADE_PLAIN))
                frames.append(r.color(0).astype(np.float64))
            out.append(frames)
        assert max(np.abs(a - b).max() for a, b in zip(*out)) <= 2e-6
        quads = [out[0][0][:, 30 * k + 2:30 * k + 28] for k in range(len(WRAPS))]
        assert all(not np.array_equal(quads[i], quads[j]) for i in range(len(WRAPS)) for j in range(i))
    finally:
        r.close()


@pytest.mark.parametrize("packed", [True, False])
def test_decoded_materials(packed):
    kept = decoder_images(np.random.default_rng(1), [(33, 17)] * 3) + decoder_images(np.random.default_rng(2), [(16, 16)] * 3)
    descs = (abi.TextureDesc * 6)(*[d for d, _ in kept])
    mats = (abi.GpuMaterial * 2)()
    for m in range(2):
        for f, _ in abi.GpuMaterial._fields_:
            if f.endswith("_index"):
                setattr(mats[m], f, 0xFFFFFFFF)
        mats[m].color_sampled_image_index, mats[m].normal_sampled_image_index = 3 * m, 3 * m + 1
        mats[m].mixmap_sampled_image_index, mats[m].normal_sampler_index = 3 * m + 2, 0
    samplers = (abi.Sampler * 1)(abi.Sampler(4 if packed else 0, 4, 2, 2))
    r = rosy_amd.Renderer(device=0)
    try:
        assert rosy_amd.lib().rsy_set_materials(r.ctx, mats, 2, descs, 6, samplers, 1) == abi.RSY_OK
        r.neural_init(latent_size=16, region=4, batch=2048)
        assert r.neural_stats().n_eligible == 2
        assert r.packed_materials()[0] == (2 if packed else 0)
    finally:
        r.close()
