"""Exact binning in one pass (fixed queue regions) at its edges: blocks whose
triangles touch few tiles, exactly 256, and more; tiles that overflow their
region (gathered by the resolve pass), and the two-pass frames that follow a
frame with many such entries.  Every frame is the oracle's, bit for bit, and
the counts are the exact ones under every route."""
import numpy as np
import pytest

import oracle as O
import rast as R
import scenes as S
from scene_util import mesh, screen_camera

pytestmark = pytest.mark.gpu


def pixel_triangles(rng, n, x0, y0, x1, y1, size, width, height):
    """n triangles with corners in the given pixel rectangle, about `size` pixels wide."""
    cx, cy = rng.uniform(x0, x1, n), rng.uniform(y0, y1, n)
    pts = []
    for k in range(n):
        z = -rng.uniform(2, 6)
        # corner order so that the triangle faces the camera
        a = rng.uniform(0, 2 * np.pi)
        for q in range(3):
            px = np.clip(cx[k] + size * np.cos(a + 2.0944 * q), x0, x1)
            py = np.clip(cy[k] + size * np.sin(a + 2.0944 * q), y0, y1)
            # w = 1 - z_view under the reference's projection
            w = 1 - z
            pts.append(((px / width * 2 - 1) * w * width / height, (1 - py / height * 2) * w, z))
    return S.Scene([mesh(pts, np.arange(3 * n).reshape(-1, 3))])


def check(r, scene, cam, opts, width, height, tile):
    vis, depth, _ = r.readback()
    ovis, odepth, _, _ = O.render(scene, cam, opts, width, height, threads=8)
    np.testing.assert_array_equal(vis, ovis)
    np.testing.assert_array_equal(depth.view(np.uint32), odepth.view(np.uint32))
    return r.debug_read(R.DEBUG_TILE_COUNTS, np.uint32)


@pytest.mark.parametrize("tile", [8, 16, 32])
@pytest.mark.parametrize("tiles_wide", [1, 16, 17])
def test_block_rectangles(tile, tiles_wide):
    W = H = 640
    edge = min(tile * tiles_wide, W) - 0.5
    scene = pixel_triangles(np.random.default_rng(tile + tiles_wide), 700, 0.25, 0.25, edge, edge, 0.6 * tile, W, H)
    cam, opts = screen_camera(), S.Opts(cull_mode=S.CULL_NONE)
    counts = {}
    with R.Renderer(W, H, tile=tile, big_threshold=1024) as r:
        r.set_tuning(0, 1024)
        r.add_scene(scene)
        for policy in (R.BIN_EXACT, R.BIN_PREVFRAME):
            r.render(cam, opts, policy)
            counts[policy] = check(r, scene, cam, opts, W, H, tile)
            st = r.stats()
            assert st["num_bin_pairs"] == counts[policy].sum()
    np.testing.assert_array_equal(counts[R.BIN_EXACT], counts[R.BIN_PREVFRAME])
    assert counts[R.BIN_EXACT].sum() >= 700  # every triangle is binned


@pytest.mark.parametrize("n", [1500, 9000])
def test_overflowing_regions_and_the_two_pass_frames_after_them(n):
    # 16,384 tiles share the queue: 1,024 entries a region; every triangle in a few tiles
    W = H = 1024
    scene = pixel_triangles(np.random.default_rng(n), n, 300.5, 300.5, 318.5, 318.5, 9.0, W, H)
    cam, opts = screen_camera(), S.Opts(cull_mode=S.CULL_NONE)
    with R.Renderer(W, H, tile=8, big_threshold=1024) as r:
        r.set_tuning(0, 1024)
        r.add_scene(scene)
        counts = []
        for _ in range(3):
            r.render(cam, opts)
            counts.append(check(r, scene, cam, opts, W, H, 8))
            st = r.stats()
            assert st["num_bin_pairs"] == counts[-1].sum()
            assert st["overflow_tiles"] == 0 and st["overflow_entries"] == 0 and st["capacity_total"] == 0
    assert counts[0].max() > 1024  # beyond a region
    np.testing.assert_array_equal(counts[0], counts[1])
    np.testing.assert_array_equal(counts[0], counts[2])
