"""Shadow-map taps at the map's edges against the oracle: maps of one texel (no pair of texels to load), two, three and a
few more, and light projections that put part of the view left of, right of, above and below the map."""
import numpy as np
import pytest

import rosy_amd
from scenes import CustomScene
from test_gpu_parity import check_frame

pytestmark = pytest.mark.gpu


def scene(size, scale, shift):
    rng = np.random.default_rng(size)
    pos = [(-1, -1, 0.2), (1, -1, 0.2), (1, 1, 0.2), (-1, 1, 0.2)]
    tri = [0, 1, 2, 0, 2, 3]
    for _ in range(12):
        x, y, z = rng.uniform(-0.9, 0.5), rng.uniform(-0.9, 0.5), rng.uniform(0.3, 0.9)
        w, h = rng.uniform(0.1, 0.5, 2)
        tri += [len(pos), len(pos) + 1, len(pos) + 2]
        pos += [(x, y, z), (x + w, y, z), (x, y + h, z)]
    light = [scale, 0, 0, 0, 0, scale, 0, 0, 0, 0, 1.0, 0, shift[0], shift[1], 0, 1.0]
    return CustomScene(pos, tri, 96, 80, shadow_projection=light, shadow_size=size)


@pytest.mark.parametrize("size", [1, 2, 3, 5, 64])
@pytest.mark.parametrize("scale,shift", [(1.0, (0, 0)), (1.7, (0, 0)), (0.9, (0.6, -0.5)), (0.9, (-0.6, 0.5))])
def test_taps_at_the_edges(size, scale, shift):
    sc = scene(size, scale, shift)
    r = rosy_amd.Renderer(device=0)
    try:
        r.load(sc)
        check_frame(r, sc)
        assert 0 < (r.visibility(0) != 0).sum()
    finally:
        r.close()
