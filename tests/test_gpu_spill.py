"""Previous-frame capacities with spill regions: tiles whose entries beyond
capacity fit their region, fill it exactly or go on to the overflow list, and
the frames after one that left many entries there (placed by passes again).
Frames are the exact ones, and the overflow counts what the tiles' counts and
capacities say."""
import numpy as np
import pytest

import rast as R
import scenes as S

pytestmark = pytest.mark.gpu

W, H = 320, 200
SKY = S.Camera(position=(0.0, 9.0, 0.0), forward=(0.0, -1.0, 0.05))
NEAR = S.Camera(position=(0.0, 20.0, -60.0), forward=(0.0, 0.3, -1.0))


def planes(r):
    vis, depth, rgba = r.readback()
    return vis, depth.view(np.uint32), rgba


def frame_and_counts(r, cam, opts, policy):
    r.render(cam, opts, policy)
    got = planes(r)
    st = r.stats()
    n = -(-W // r.tile) * -(-H // r.tile)
    counts = r.debug_read(R.DEBUG_TILE_COUNTS, np.uint32)[:n].astype(np.int64)
    caps = r.debug_read(R.DEBUG_TILE_CAPS, np.uint32)[:n].astype(np.int64)
    return got, st, counts, caps


# terrain 24: a few entries a tile; 90: hundreds, some above 512 at 32 pixels;
# 260: above 512 in most tiles, more than 32,768 entries on the list
@pytest.mark.parametrize("tile", [8, 16, 32])
@pytest.mark.parametrize("size", [24, 90, 260])
def test_overflowing_tiles(tile, size):
    scene, opts = S.Scene([S.terrain(size)]), S.Opts(cull_mode=S.CULL_NONE)
    with R.Renderer(W, H, tile=tile, big_threshold=1024) as r, R.Renderer(W, H, tile=tile, big_threshold=1024) as exact:
        for x in (r, exact):
            x.set_tuning(0, 16)  # every triangle is binned
            x.add_scene(scene)
        most = 0
        for cams in ((SKY, NEAR, NEAR), (NEAR, SKY, NEAR)):
            r.set_queue_depth(1.0, 0)
            r.render(cams[0], opts, R.BIN_EXACT, R.FLAG_NO_SHADE)
            for k, cam in enumerate(cams[1:]):
                got, st, counts, caps = frame_and_counts(r, cam, opts, R.BIN_PREVFRAME)
                exact.render(cam, opts, R.BIN_EXACT)
                for a, b in zip(got, planes(exact)):
                    np.testing.assert_array_equal(a, b)
                over = np.maximum(counts - caps, 0)
                assert st["overflow_entries"] == over.sum()
                assert st["overflow_tiles"] == np.count_nonzero(over)
                most = max(most, int(over.max()))
        assert most > 0


def test_frames_after_a_camera_cut():
    """The frame after a cut overflows its spill regions; later exact frames of
    the same view and further previous-frame ones stay the exact frame."""
    scene, opts = S.Scene([S.terrain(260)]), S.Opts(cull_mode=S.CULL_NONE)
    with R.Renderer(W, H, tile=32, big_threshold=1024) as r:
        r.set_tuning(0, 16)
        r.add_scene(scene)
        r.render(NEAR, opts, R.BIN_EXACT)
        want = planes(r)
        r.set_queue_depth(1.0, 0)
        r.render(SKY, opts, R.BIN_EXACT, R.FLAG_NO_SHADE)
        for policy in (R.BIN_PREVFRAME, R.BIN_EXACT, R.BIN_PREVFRAME, R.BIN_EXACT):
            r.render(NEAR, opts, policy)
            for a, b in zip(planes(r), want):
                np.testing.assert_array_equal(a, b)
