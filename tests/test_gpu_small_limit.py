"""Triangles on both sides of the line between the two ways a tile rasterizes its
queue (as items, or one pixel per lane from half the tile's pixels or from
small_limit, whichever is more): ranges one pixel row or column around half a
tile and around the whole of it, and limits around both.  Whole tiles, and
quarters of 32-pixel tiles in launches of few tiles; against the oracle."""
import numpy as np
import pytest

import oracle as O
import rast as R
import scenes as S
from scene_util import mesh, screen_camera, turned
from test_gpu_fixed_regions import pixel_triangles

pytestmark = pytest.mark.gpu


def around_half(tile, width, height):
    """Right triangles whose pixel ranges hold about half a tile or all of it, two a tile."""
    rng = np.random.default_rng(tile)
    pts = []
    sizes = [(w, h) for w in (tile // 2 - 1, tile // 2, tile // 2 + 1, tile - 1, tile) for h in (tile // 2, tile - 1, tile)]
    for ty in range(height // tile):
        for tx in range(width // tile):
            for _ in range(2):
                w, h = sizes[rng.integers(len(sizes))]
                x0, y0 = tx * tile + 0.25, ty * tile + 0.25
                z = -rng.uniform(2, 6)
                for px, py in ((x0, y0), (x0, y0 + h - 0.5), (x0 + w - 0.5, y0)):
                    c = 1 - z
                    pts.append(((px / width * 2 - 1) * c * width / height, (1 - py / height * 2) * c, z))
    return S.Scene([mesh(pts, np.arange(len(pts)).reshape(-1, 3))])


@pytest.mark.parametrize("kind", ["grid", "random"])
@pytest.mark.parametrize("tile,size", [(8, 256), (16, 384), (32, 768), (32, 320)])  # 320: quarters
def test_limits_around_half_a_tile(kind, tile, size):
    part = 16 if size == 320 else tile
    half, full = part * part // 2, part * part
    if kind == "grid":
        scene = around_half(part, size, size)
    else:
        scene = turned(pixel_triangles(np.random.default_rng(tile), 1500, 0.25, 0.25, size - 0.25, size - 0.25,
                                       0.9 * part, size, size))
    cam, opts = screen_camera(), S.Opts(cull_mode=S.CULL_NONE)
    ovis, odepth, _, _ = O.render(scene, cam, opts, size, size, threads=8, want_rgba=False)
    assert np.count_nonzero(ovis != R.VIS_NONE) > size * size // 8
    with R.Renderer(size, size, tile=tile, big_threshold=1024) as r:
        r.add_scene(scene)
        for limit in sorted({0, half - 1, half, half + 1, half + part, full - 1, full, 1024}):
            r.set_tuning(0, min(limit, 1024))
            r.render(cam, opts)
            vis, depth, _ = r.readback()
            np.testing.assert_array_equal(vis, ovis, err_msg=f"limit {limit}")
            np.testing.assert_array_equal(depth.view(np.uint32), odepth.view(np.uint32), err_msg=f"limit {limit}")
