"""Views of a scene large enough that vertex chunks are transformed only for the
views they may be in, frames whose unread records are left out, and frames without shading, which form no attributes: the frame, and the debug
buffers, which are completed on demand, hold what the oracle does."""
import copy

import numpy as np
import pytest

import oracle as O
import rast as R
import scenes as S

pytestmark = pytest.mark.gpu

N = 400  # 160,801 vertices: 1,257 chunks, 17,598 to transform for 14 views
W, H = 320, 200
CAMERAS = [S.Camera(position=(0.0, 9.0, 0.0), forward=(0.0, -0.2, 1.0)),
           S.Camera(position=(0.0, 9.0, 0.0), forward=(0.7, -0.1, -0.7)),
           S.Camera(position=(0.0, 20.0, -60.0), forward=(0.0, -0.3, 1.0)),
           S.Camera(position=(0.0, 9.0, 0.0), forward=(0.0, 1.0, 0.05))]  # the sky: nothing in view


def scene(kind):
    """A terrain that reaches out of every view, and a sphere with its own world matrix."""
    t = S.terrain(N)
    if kind == "shuffled":  # every chunk used by triangles from everywhere
        tri = t.indices.reshape(-1, 3)
        t.indices = np.ascontiguousarray(tri[np.random.default_rng(3).permutation(len(tri))]).ravel()
    elif kind == "strip":
        w = N + 1
        rows = []
        for j in range(N):
            top = np.arange(j * w, j * w + w, dtype=np.uint32)
            row = np.stack([top, top + w], 1).ravel()
            rows += [row[:1], row, row[-1:]]
        t.indices, t.topology = np.concatenate(rows), S.TOPO_STRIP
    ball = S.uv_sphere(32, 16)
    ball.world = S.world_matrix((2.0, 8.0, 6.0), (0.3, 0.2, 0.1), 1.5)
    return S.Scene([t, ball])


def check_frame(got, sc, cam, opts):
    vis, depth, rgba, _ = O.render(sc, cam, opts, W, H, threads=8)
    np.testing.assert_array_equal(got[0], vis)
    np.testing.assert_array_equal(got[1].view(np.uint32), depth.view(np.uint32))
    if len(got) > 2:
        d = np.abs(got[2].view(np.uint8).astype(int) - rgba.view(np.uint8).astype(int))
        assert d.max() <= 1


def check_debug(r, sc, cam, opts, attributes=True, first_mesh=0):
    both = [O.vertex_transform(sc, cam, W, H, k) for k in range(len(sc.meshes))]
    opos, oattr = (np.concatenate([b[q] for b in both]) for q in range(2))
    pos = r.debug_read(R.DEBUG_VERTEX_POS, np.uint32).reshape(-1, 4)
    np.testing.assert_array_equal(pos, np.ascontiguousarray(opos.astype(np.float32)).view(np.uint32))
    if attributes:
        attr = r.debug_read(R.DEBUG_VERTEX_ATTR, np.float32).reshape(-1, 12)
        inv_w = oattr[:, 14:15].astype(np.float32)
        want = np.concatenate([(oattr[:, :11].astype(np.float32) * inv_w).astype(np.float32), inv_w], axis=1)
        got = np.ascontiguousarray(attr[:, [0, 1, 3, 4, 5, 6, 7, 8, 9, 10, 11, 2]])
        np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    flags, orec = O.setup(sc, cam, opts.cull_mode, W, H)
    np.testing.assert_array_equal(r.debug_read(R.DEBUG_TRI_ALIVE, np.uint8), flags)
    live = flags.astype(bool)
    rec = r.debug_read(R.DEBUG_TRI_RECORDS, np.uint32).reshape(-1, 16)[live]
    # the mesh entry counts over the launch (the views before this one have two meshes each)
    mesh = np.repeat(np.arange(len(sc.meshes)), [m.num_triangles for m in sc.meshes])[live]
    np.testing.assert_array_equal(rec[:, 15] & 0x7FFFFFFF, mesh + first_mesh)
    np.testing.assert_array_equal(np.ascontiguousarray(rec[:, [0, 1, 2, 3, 4, 5, 6, 9, 8, 7, 10, 11]]),
                                  np.ascontiguousarray(orec[live]).view(np.uint32))


@pytest.mark.parametrize("kind", ["list", "strip", "shuffled"])
def test_frames_and_debug_buffers(kind):
    sc, opts = scene(kind), S.Opts()
    with R.Renderer(W, H) as r:
        r.add_scene(sc)
        for k, cam in enumerate(CAMERAS):  # other chunks in view each time: nothing stale is read
            r.render(cam, opts, R.BIN_EXACT, 0 if k != 1 else R.FLAG_NO_SHADE)
            check_frame(r.readback(rgba=k != 1)[:3 if k != 1 else 2], sc, cam, opts)
            check_debug(r, sc, cam, opts)


@pytest.mark.parametrize("kind", ["list", "strip", "shuffled"])
def test_views_of_one_scene(kind):
    sc, opts = scene(kind), S.Opts()
    owner = R.Renderer(W, H)
    owner.add_scene(sc)
    rs = [owner] + [owner.view(W, H) for _ in range(13)]  # a round of eight entries and a part
    try:
        for turn in range(2):
            cams = [CAMERAS[(k + turn) % len(CAMERAS)] for k in range(len(rs))]
            R.render_batch([(r, cam, opts, R.BIN_EXACT, 0) for r, cam in zip(rs, cams)])
            for r, cam in list(zip(rs, cams))[:5] + list(zip(rs, cams))[12:]:
                check_frame(r.readback(), sc, cam, opts)
            check_debug(rs[13], sc, cams[13], opts, attributes=False, first_mesh=26)
    finally:
        for r in rs[:0:-1]:
            r.close()
        owner.close()


def test_debug_buffers_are_the_frame_s_after_the_scene_changes():
    sc, opts, cam = scene("list"), S.Opts(), CAMERAS[0]
    drawn = copy.deepcopy(sc)
    for change in ("world", "destroy"):
        with R.Renderer(W, H) as r:
            handles = [r.add_mesh(m) for m in sc.meshes]
            r.render(cam, opts)
            if change == "world":
                m = np.ascontiguousarray(S.world_matrix((9.0, 9.0, 9.0), (0, 0, 0), 1.0), np.float32)
                R.check(R.lib().rast_mesh_set_world(handles[1], m.ctypes.data), "rast_mesh_set_world")
            else:
                R.check(R.lib().rast_mesh_destroy(handles[1]), "rast_mesh_destroy")
            check_debug(r, drawn, cam, opts)
