"""A first frame that leaves more entries beyond its fixed regions than the
overflow list holds is drawn again by two passes; it and the frames after it,
through the return to one pass, are the oracle's."""
import numpy as np
import pytest

import rast as R
import scenes as S
from scene_util import screen_camera, turned
from test_gpu_fixed_regions import check, pixel_triangles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("policy", [R.BIN_EXACT, R.BIN_PREVFRAME])
def test_first_frame_beyond_the_overflow_list(policy):
    # 64 tiles of 16,384 entries each, most of them wanted by 60,000 triangles
    W = H = 64
    scene = turned(pixel_triangles(np.random.default_rng(5), 60000, 0.5, 0.5, 63.5, 63.5, 45.0, W, H))
    cam, opts = screen_camera(), S.Opts(cull_mode=S.CULL_NONE)
    away = S.Camera(position=(0.0, 0.0, 400.0), forward=cam.forward, fov_deg=cam.fov_deg, near_z=cam.near_z, far_z=1e4)
    with R.Renderer(W, H, tile=8, big_threshold=1024) as r:
        r.set_tuning(0, 1024)
        r.set_queue_depth(1.0, 0)
        r.add_scene(scene)
        r.render(cam, opts)
        counts = check(r, scene, cam, opts, W, H, 8)
        assert np.maximum(counts.astype(np.int64) - 16384, 0).sum() > 1 << 20
        assert r.stats()["rerenders"] == 1
        assert np.count_nonzero(r.readback()[0] != R.VIS_NONE) > W * H // 2
        for _ in range(20):  # they fit
            r.render(away, opts, policy)
        check(r, scene, away, opts, W, H, 8)
        assert r.stats()["rerenders"] == 1
        r.render(cam, opts, policy)
        again = check(r, scene, cam, opts, W, H, 8)
        np.testing.assert_array_equal(counts, again)
        assert r.stats()["num_bin_pairs"] == counts.sum()
