"""The decoder at latents of every size that a half holds, with first-layer weights small enough that hidden values stay
near one: stored FP8 codes span the same range whatever their scale, so the scale has to come before the hidden values
are split into halves."""
import numpy as np
import pytest

import oracle
import rosy_amd
from rosy_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weights", [0, abi.NEURAL_WEIGHTS_FP8], ids=["fp16", "fp8"])
@pytest.mark.parametrize("size", [1.0, 300.0, 4000.0, 60000.0])
def test_decode(size, weights):
    L, n = 16, 2
    rng = np.random.default_rng(int(size))
    scene = rosy_amd.Scene(3, seed=2, total_triangles=20000, n_meshes=24, width=64, height=64, shadow_size=64,
                           texture_size=16, n_materials=n)
    r = rosy_amd.Renderer(device=0)
    try:
        r.load(scene)
        r.neural_init(latent_size=L, weights=weights, psnr_threshold=0.0)
        lat = (size * rng.uniform(-1, 1, (n, L, L, 8))).astype(np.float32)
        mlp = np.zeros(583, np.float32)
        mlp[:320] = rng.uniform(-0.5, 0.5, 320)
        mlp[:320].reshape(32, 10)[:, :8] /= size
        # (the positional weights and the biases are as small as the others: one scale a layer)
        mlp[:320].reshape(32, 10)[:, 8:] /= size
        mlp[352:576] = rng.uniform(-0.1, 0.1, 224)
        mlp[576:] = 0.5
        r.neural_set_params(lat, mlp)
        r.neural_evaluate()
        material, uv = rng.integers(0, n, 2000), rng.uniform(-1, 2, (2000, 2)).astype(np.float32)
        got = r.neural_decode(material, uv)
        p = oracle.NeuralParams(np.arange(n), lat.astype(np.float16).astype(np.float32), r.neural_inference_mlp(), np.ones(n))
        want = oracle.nm_decode(p, material, uv)
        # hidden values up to 4: weights of a footprint known to 16 * 2^-23 (2e-6) between cells up to 2 apart, eight
        # times 0.5 of them, and 2^-21 of the sums: 2e-5; 32 of them times 0.1 into an output: 7e-5
        assert np.abs(got - want).max() <= 1e-4, np.abs(got - want).max()
        assert ((want > 0.01) & (want < 0.99)).mean() > 0.5
    finally:
        r.close()
        scene.close()
