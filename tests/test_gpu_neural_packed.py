"""A training step on materials sampled as one packed image against the same maps sampled one by one (their normal map's
minification filter differs, which single-level images have no use for): the same targets to the bit, so the same loss
and the same MLP after one step, at map sizes around the 4 x 4 texel tile and down to one texel."""
import numpy as np
import pytest

import rosy_amd
from rosy_amd import abi
from test_gpu_neural_eval import images

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(1, 1), (3, 2), (4, 4), (5, 7), (33, 17), (64, 64)])
def test_one_step(size):
    rng = np.random.default_rng(size[0])
    kept = images(rng, [size] * 3) + images(rng, [(16, 16)] * 3)
    descs = (abi.TextureDesc * 6)(*[d for d, _ in kept])
    scene = rosy_amd.Scene(3, seed=2, total_triangles=20000, n_meshes=24, width=64, height=64, shadow_size=64,
                           texture_size=16, n_materials=2)
    out = []
    for packed in (True, False):
        r = rosy_amd.Renderer(device=0)
        try:
            r.load(scene)
            samplers = (abi.Sampler * 2)(abi.Sampler(4, 4, 2, 2), abi.Sampler(4 if packed else 0, 4, 2, 2))
            mats = (abi.GpuMaterial * 2)(scene.s.materials[0], scene.s.materials[1])
            for m in range(2):
                mats[m].color_sampler_index = mats[m].metallic_sampler_index = mats[m].mixmap_sampler_index = 0
                mats[m].normal_sampler_index = 1
            assert rosy_amd.lib().rsy_set_materials(r.ctx, mats, 2, descs, 6, samplers, 2) == 0
            r.neural_init(latent_size=16, region=4, batch=2048)
            assert r.neural_stats().n_eligible == 2
            loss = r.neural_train(1)
            out.append((np.asarray(loss), r.neural_params()[1]))
        finally:
            r.close()
    scene.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    assert float(np.ravel(out[0][0])[0]) > 0
