"""Training steps at the sizes where their kernel's branches meet: region sides from 2 to 32 cells (fewer cells than
threads, and several cells a thread), sample counts that leave part of a 256-sample chunk empty or take several,
maps of one extent and of different ones, odd extents whose footprints wrap around.

A step from zero moments moves each parameter by lr * g / (|g| + eps'), so the first step's direction is the sign of
the FP64 gradient wherever that is not itself within rounding of zero; the loss is compared directly."""
import ctypes as C

import numpy as np
import pytest

import oracle
import rosy_amd
from rosy_amd import abi

pytestmark = pytest.mark.gpu
MASK = (1 << 64) - 1


def mix(z):
    """SplitMix64's finaliser, which numbers the samples (Steele, Lea and Flood's generator)."""
    z = (z + 0x9E3779B97F4A7C15) & MASK
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & MASK
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & MASK
    return z ^ (z >> 31)


def first_step_samples(seed, n_slots, latent, region, batch):
    """(slot, u, v) of every sample of step 0."""
    across = latent // region
    regions = n_slots * across * across
    wgs = min(batch // 256, regions)
    per = -(-batch // wgs)
    shift = mix(seed ^ mix(0x5BD1E995))
    key = mix((seed + 0x632BE59BD9B4E019) & MASK)
    f = np.float32
    slot, uv = [], []
    for b in range(wgs):
        r = b % regions
        reg = ((r // n_slots) * 2654435761) & (across * across - 1)
        rx = (reg % across) * region + (shift & (region - 1))
        ry = (reg // across) * region + ((shift >> 32) & (region - 1))
        for q in range(per):
            h = mix((key + (b << 32) + q) & MASK)
            at = [float(f((x & 0xFFFFFFFF) >> 8) / f(16777216)) * (region - 1) for x in (h, h >> 32)]
            slot.append(r % n_slots)
            uv.append(((rx + at[0] + 0.5) / latent, (ry + at[1] + 0.5) / latent))
    return np.array(slot), np.array(uv), per * wgs


def maps(rng, sizes):
    out = []
    for (w, h), fmt, ch in zip(sizes, (abi.TEX_RGBA8_SRGB, abi.TEX_RG8_UNORM, abi.TEX_RG8_SRGB), (4, 2, 2)):
        px = rng.integers(0, 256, (h, w, ch), dtype=np.uint8)
        if ch == 4:
            px[..., 3] = 255
        out.append((abi.TextureDesc(w, h, fmt, 1, px.ctypes.data), px))
    return out


@pytest.mark.parametrize("region,latent,batch,sizes", [
    (2, 8, 1024, ((16, 16),) * 3),
    (8, 16, 512, ((33, 17),) * 3),
    (16, 16, 768, ((64, 64), (31, 20), (64, 64))),  # one region a slot: several chunks, the last one short
    (16, 32, 2048, ((5, 7), (5, 7), (64, 3))),
    (32, 32, 512, ((50, 50),) * 3),
])
def test_first_step(region, latent, batch, sizes):
    rng = np.random.default_rng(region * 1000 + batch)
    scene = rosy_amd.Scene(3, seed=2, total_triangles=20000, n_meshes=24, width=64, height=64, shadow_size=64,
                           texture_size=16, n_materials=2)
    r = rosy_amd.Renderer(device=0)
    try:
        r.load(scene)
        kept = maps(rng, sizes) + maps(rng, sizes)
        descs = (abi.TextureDesc * 6)(*[d for d, _ in kept])
        assert rosy_amd.lib().rsy_set_materials(r.ctx, scene.s.materials, 2, descs, 6, scene.s.samplers,
                                                scene.s.n_samplers) == 0
        seed, lr = 77, 1e-3
        r.neural_init(latent_size=latent, region=region, batch=batch, seed=seed, lr_mlp=lr, lr_latent=lr)
        lat = rng.uniform(-0.8, 0.8, (2, latent, latent, 8)).astype(np.float32)
        mlp = rng.uniform(-0.5, 0.5, 583).astype(np.float32)
        r.neural_set_params(lat, mlp)
        loss = r.neural_train(1)
        lat1, mlp1 = r.neural_params()

        slot, uv, n = first_step_samples(seed, 2, latent, region, batch)
        want = np.array([np.concatenate([np.asarray(oracle.sample_texture(kept[3 * s + k][0], None, u, v))[:c]
                                         for k, c in enumerate((3, 2, 2))]) for s, (u, v) in zip(slot, uv)])
        p = oracle.NeuralParams(np.arange(2), lat, mlp)
        loss_o, gm, gl, _ = oracle.nm_gradients(p, slot, uv.astype(np.float32), want.astype(np.float32))
        # sample coordinates are FP32: 1e-6 of a cell or texel, against targets and features of slope <= 1 a texel
        # or cell, moves a sample's error by a few 1e-6 of its size (0.3): the loss to 1e-4 relative
        assert abs(loss[0] - loss_o) <= 1e-4 * loss_o, (loss[0], loss_o)
        # the update's direction and size where the gradient is well away from its rounding (1e-3 of the largest)
        for before, after, g in ((mlp, mlp1, gm), (lat, lat1, gl)):
            clear = np.abs(g) > 1e-3 * np.abs(g).max()
            step = (after.astype(np.float64) - before)[clear]
            ideal = -lr * g[clear] / (np.abs(g[clear]) + 1e-8)
            assert clear.sum() > 0.2 * (g != 0).sum()
            # |step - ideal|: one FP32 rounding of a parameter below 1 (6e-8) and the gradient's error through
            # eps / (|g| + eps)^2, bounded by 2 % of the step for gradients known to 1 %
            assert np.abs(step - ideal).max() <= 1e-7 + 0.02 * lr, np.abs(step - ideal).max()
            untouched = g == 0
            if before is lat:  # cells outside every footprint keep their latents
                assert np.array_equal(after[untouched], before[untouched])
    finally:
        r.close()
        scene.close()
