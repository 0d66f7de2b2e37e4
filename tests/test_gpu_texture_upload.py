"""Many images in one upload, bit-exact against the oracle: chains of every length around the 64-texel tile and the
six levels that one launch builds, BC7 images with several given levels between them, and the alpha test where a
single texel of an image is not opaque."""
import numpy as np
import pytest

import oracle
import rosy_amd
from oracle import textures as tx
from rosy_amd import abi
from test_gpu_neural_eval import images
from test_gpu_textures import random_blocks, read, renderer, upload  # noqa: F401

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (1, 130), (63, 64), (64, 64), (65, 127), (128, 129), (200, 3), (257, 130)]


def test_chains_of_many_sizes_in_one_upload(renderer):  # noqa: F811
    rng = np.random.default_rng(11)
    ups, want = [], []
    for k, (w, h) in enumerate(SIZES):
        for fmt, ch, srgb in ((abi.TEX_RGBA8_SRGB, 4, True), (abi.TEX_RG8_UNORM, 2, False)):
            px = rng.integers(0, 256, (h, w, ch), dtype=np.uint8)
            if ch == 4:
                px[rng.random((h, w)) < 0.2, 3] = 0
            ups.append((w, h, fmt, abi.MIPS_BUILD, px.tobytes()))
            want.append(tx.mip_chain(px, srgb))
        given = min(3, max(w, h).bit_length())
        sizes = [(max(1, w >> l), max(1, h >> l)) for l in range(given)]
        blocks = [random_blocks(rng, ((lw + 3) // 4) * ((lh + 3) // 4)).tobytes() for lw, lh in sizes]
        ups.append((w, h, abi.TEX_BC7_UNORM, given, b"".join(blocks)))
        want.append([oracle.bc7_decode(b, lw, lh) for b, (lw, lh) in zip(blocks, sizes)])
    assert upload(renderer, ups) == abi.RSY_OK
    for t, (w, h, fmt, _, _) in enumerate(ups):
        assert len(want[t]) == 3 or len(want[t]) == max(w, h).bit_length()
        for l, level in enumerate(want[t]):
            got = read(renderer, t, l, w, h, level.shape[2])
            assert np.array_equal(got, level), (t, w, h, l)


@pytest.mark.parametrize("size", [(1, 1), (65, 17), (300, 220)])
def test_one_clear_texel_is_found(size):
    rng = np.random.default_rng(12)
    w, h = size
    scene = rosy_amd.Scene(3, seed=2, total_triangles=20000, n_meshes=24, width=64, height=64, shadow_size=64,
                           texture_size=16, n_materials=2)
    r = rosy_amd.Renderer(device=0)
    try:
        r.load(scene)
        kept = images(rng, [size] * 3) + images(rng, [(16, 16)] * 3)
        albedo = kept[0][1]
        descs = (abi.TextureDesc * 6)(*[d for d, _ in kept])
        for y, x, a, eligible in ((0, 0, 255, 2), (h - 1, w - 1, 254, 1), (0, 0, 0, 1), (h // 2, w // 2, 254, 1)):
            albedo[..., 3] = 255
            albedo[y, x, 3] = a
            assert rosy_amd.lib().rsy_set_materials(r.ctx, scene.s.materials, 2, descs, 6, scene.s.samplers,
                                                    scene.s.n_samplers) == 0
            r.neural_init(latent_size=4, region=2)
            assert r.neural_stats().n_eligible == eligible, (y, x, a)
    finally:
        r.close()
        scene.close()
