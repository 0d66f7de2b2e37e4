"""The decoder's evaluation over texel tiles: PSNR per material against the FP64 decoder and sampler at every texel
centre of the albedo map, at sizes around the 64 x 16 texel tile, with maps of one extent (texels read directly) and of
different extents (sampled bilinearly), and latent grids coarser and finer than the maps."""
import ctypes as C

import numpy as np
import pytest

import oracle
import rosy_amd
from rosy_amd import abi

pytestmark = pytest.mark.gpu

SIZES = [  # albedo, normal, metallic-roughness (width, height), latent cells per side
    ((1, 1), (1, 1), (1, 1), 4),
    ((63, 15), (63, 15), (63, 15), 8),
    ((64, 16), (64, 16), (64, 16), 32),
    ((65, 17), (65, 17), (65, 17), 16),
    ((130, 33), (130, 33), (130, 33), 64),
    ((64, 64), (32, 32), (64, 64), 16),
    ((70, 20), (70, 20), (33, 7), 32),
]


def images(rng, sizes):
    """One material's three maps: descriptors and the texels they point at."""
    out = []
    for (w, h), fmt, ch in zip(sizes, (abi.TEX_RGBA8_SRGB, abi.TEX_RG8_UNORM, abi.TEX_RG8_SRGB), (4, 2, 2)):
        px = rng.integers(0, 256, (h, w, ch), dtype=np.uint8)
        if ch == 4:
            px[..., 3] = 255  # opaque: eligible
        out.append((abi.TextureDesc(w, h, fmt, 1, px.ctypes.data), px))
    return out


def tolerance(mse):
    """dB: the decoder is within 2e-5 and the target within 1e-5 of FP64, so |d mse| <= 2 e sqrt(mse) + e^2."""
    e = 3e-5
    return 10 / np.log(10) * (2 * e / np.sqrt(mse) + e * e / mse) + 1e-5


@pytest.mark.parametrize("weights", [abi.NEURAL_WEIGHTS_FP16, abi.NEURAL_WEIGHTS_FP8])
@pytest.mark.parametrize("sizes", SIZES, ids=lambda s: "x".join(f"{w}_{h}" for w, h in s[:3]) + f"_L{s[3]}")
def test_psnr_over_tiles(sizes, weights):
    *maps, latent = sizes
    rng = np.random.default_rng(sum(w * 31 + h for w, h in maps) + latent)
    scene = rosy_amd.Scene(3, seed=2, total_triangles=20000, n_meshes=24, width=64, height=64, shadow_size=64,
                           texture_size=16, n_materials=2)
    r = rosy_amd.Renderer(device=0)
    try:
        r.load(scene)
        # material 0: the maps under test; material 1: 16 x 16 maps of its own
        kept = images(rng, maps) + images(rng, [(16, 16)] * 3)
        descs = (abi.TextureDesc * 6)(*[d for d, _ in kept])
        assert rosy_amd.lib().rsy_set_materials(r.ctx, scene.s.materials, 2, descs, 6, scene.s.samplers,
                                                scene.s.n_samplers) == 0
        r.neural_init(latent_size=latent, region=2, weights=weights, psnr_threshold=0.0)
        lat = rng.uniform(-0.6, 0.8, (2, latent, latent, 8)).astype(np.float32)
        r.neural_set_params(lat, rng.uniform(-0.5, 0.5, 583).astype(np.float32))
        got = r.neural_evaluate()
        p = oracle.NeuralParams(np.arange(2), lat.astype(np.float16).astype(np.float32), r.neural_inference_mlp())
        for m in range(2):
            d = [x for x, _ in kept[3 * m:3 * m + 3]]
            w, h = d[0].width, d[0].height
            uv = np.array([((x + 0.5) / w, (y + 0.5) / h) for y in range(h) for x in range(w)])
            want = np.array([np.concatenate([np.asarray(oracle.sample_texture(t, None, u, v))[:n]
                                             for t, n in zip(d, (3, 2, 2))]) for u, v in uv])
            dec = oracle.nm_decode(p, np.full(len(uv), m), uv)
            mse = np.mean((dec - want) ** 2)
            assert abs(got[m] + 10 * np.log10(mse)) <= tolerance(mse), (m, got[m], mse)
    finally:
        r.close()
        scene.close()
