"""The raster's tasks (row segments of staged records) against the oracle, bit for bit: boxes one pixel short of, at and past
a segment's and a tile's width, and bins holding one record, a whole word of 64 tasks, a whole chunk of 128
records or an item of 256, each less or more one, with one and four samples and every bin size."""
import numpy as np
import pytest

import oracle
import rosy_amd
from rosy_amd import abi
from scenes import CustomScene

pytestmark = pytest.mark.gpu

W, H = 150, 70


def boxes_scene(kind):
    """Right triangles over boxes of w x h pixels at (x, y), reverse-Z depths drawn at random."""
    rng = np.random.default_rng(5)
    if kind == "widths":
        boxes = [(x, y, w, h) for w in (1, 7, 8, 9, 15, 16, 17, 23, 24, 25, 31, 32, 33, 63, 64, 65)
                 for x, y, h in ((0, 0, 1), (3, 5, 7), (37, 30, 33), (64, 2, 64))]
    else:  # `kind` records of one pixel in one bin, and one large one behind them
        boxes = [(x % 8, x // 8 % 8, 1, 1) for x in range(kind)] + [(0, 0, 40, 40)]
    pos, tri = [], []
    for i, (x, y, w, h) in enumerate(boxes):
        z = rng.uniform(0.2, 0.9) if i < len(boxes) - 1 else 0.1
        x0, x1 = x / W * 2 - 1, (x + w + 0.25) / W * 2 - 1
        y0, y1 = y / H * 2 - 1, (y + h + 0.25) / H * 2 - 1
        tri += [3 * i, 3 * i + 1, 3 * i + 2]
        flip = bool(rng.integers(0, 2))
        pos += [(x0, y0, z), (x1, y0, z), (x0, y1, z)] if flip else [(x1, y1, z), (x0, y1, z), (x1, y0, z)]
    return CustomScene(pos, tri, W, H)


@pytest.mark.parametrize("samples,tile", [(1, 8), (1, 16), (1, 32), (1, 64), (4, 32)])
@pytest.mark.parametrize("kind", ["widths", 1, 63, 64, 65, 127, 128, 129, 255, 256, 257])
def test_tasks(kind, samples, tile):
    sc = boxes_scene(kind)
    rs = sc.s.raster_state
    rs.msaa_samples, rs.tile_size = samples, tile
    r = rosy_amd.Renderer(device=0)
    try:
        r.load(sc)
        r.render(sc.frame_desc(abi.SHADE_PLAIN))
        vp = sc.camera_views()[0].view_projection[:]
        want = oracle.raster_view_msaa(sc, vp, W, H, rs) if samples == 4 else oracle.raster_view(sc, vp, W, H, False, rs)[0]
        got = r.visibility(0)
        assert np.array_equal(got, want), f"{int((got != want).sum())} words differ"
        assert (want != 0).sum() > 500 * samples
    finally:
        r.close()
