"""The shading instances with 64-bit record addresses, which only scenes of more
than 89 million vertices or 67 million triangles need, on scenes small enough to
test: the frame is the same bytes, for single frames and views of one launch,
each sampling mode, a mesh without maps, one map, four maps of two sizes and of
one, and triangles that are shaded in the reference's order."""
import numpy as np
import pytest

import rast as R
import scenes as S

pytestmark = pytest.mark.gpu

W, H = 333, 217
CAMERAS = [S.orbit_camera(0.3 * k, 0.2, 3.0) for k in range(3)]


def scene():
    maps = S.noise_maps(64, S.SEED_BASE + 5)
    small = S.noise_maps(32, S.SEED_BASE + 6)
    meshes = []
    for k, tex in enumerate((None, [maps[0], None, None, None], [maps[0], small[1], maps[2], small[3]], maps)):
        m = S.uv_sphere(48, 24, 0.8)
        m.world = S.world_matrix((0.9 * k - 1.3, 0.2 * k, -0.3 * k), (0.1 * k, 0.2, 0.0), 1.0)
        m.textures = tex
        meshes.append(m)
    ground = S.terrain(24, 8.0, 0.5, 3, 9, 1.0)  # reaches behind the camera plane
    ground.textures = maps
    return S.Scene(meshes + [ground])


@pytest.mark.parametrize("sample", [S.SAMPLE_POINT, S.SAMPLE_LINEAR])
@pytest.mark.parametrize("visualisation", [0, 1, 2])
def test_single_frames(sample, visualisation):
    opts = S.Opts(sample_state=sample, visualisation=visualisation, cull_mode=S.CULL_NONE)
    with R.Renderer(W, H) as r:
        r.add_scene(scene())
        for cam in CAMERAS:
            got = []
            for flags in (0, R.FLAG_FAR, R.FLAG_FAR | R.FLAG_GRAPH):
                r.render(cam, opts, R.BIN_EXACT, flags)
                got.append(r.readback())
            if visualisation != 1:  # (so near, depths are all black)
                assert np.unique(got[0][2]).size > 100
            for other in got[1:]:
                for a, b in zip(got[0], other):
                    np.testing.assert_array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("sample", [S.SAMPLE_POINT, S.SAMPLE_LINEAR])
def test_views_of_one_launch(sample):
    opts = S.Opts(sample_state=sample, cull_mode=S.CULL_NONE)
    owner = R.Renderer(W, H)
    owner.add_scene(scene())
    rs = [owner, owner.view(W, H), owner.view(W - 60, H + 11)]
    try:
        got = []
        for flags in ((0, 0, 0), (R.FLAG_FAR,) * 3, (0, R.FLAG_FAR, 0)):  # also beside one another
            R.render_batch([(r, cam, opts, R.BIN_EXACT, f) for r, cam, f in zip(rs, CAMERAS, flags)])
            got.append([r.readback() for r in rs])
        for other in got[1:]:
            for want, have in zip(got[0], other):
                for a, b in zip(want, have):
                    np.testing.assert_array_equal(a.view(np.uint32), b.view(np.uint32))
    finally:
        for r in rs[::-1]:
            r.close()
