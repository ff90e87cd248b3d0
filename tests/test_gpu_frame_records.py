"""What a frame itself formed, as it left it (a plain debug read forms it anew):
the setup record of every triangle in the picture, the positions and attributes
of their vertices and of the screen list's, are this frame's and no other's."""
import numpy as np
import pytest

import oracle as O
import rast as R
import scenes as S
from test_gpu_chunk_cull import H, W, scene

pytestmark = pytest.mark.gpu

PATH = S.camera_path(S.SEED_BASE + 3, 200)
CAMERAS = [PATH[0], S.Camera(position=(0.0, 20.0, -60.0), forward=(0.0, 0.3, -1.0)), PATH[60], PATH[120]]


def indices(sc):
    """Global vertex indices of all triangles, in ID order."""
    out, base = [], 0
    for m in sc.meshes:
        ix = m.indices.astype(np.int64)
        if m.topology == S.TOPO_LIST:
            t = ix[: ix.size // 3 * 3].reshape(-1, 3)
        else:
            k = np.arange(ix.size - 2)
            t = np.stack([ix[k], ix[k + 1 + k % 2], ix[k + 2 - k % 2]], 1)
        out.append(t + base)
        base += len(m.verts)
    return np.concatenate(out)


def check(r, sc, cam, opts, attributes=True, first_mesh=0):
    vis = r.readback(depth=False, rgba=False)[0]
    ovis, _, _, _ = O.render(sc, cam, opts, W, H, threads=8, want_rgba=False)
    np.testing.assert_array_equal(vis, ovis)
    big = r.debug_read(R.DEBUG_BIG_LIST, np.uint32)[1:]
    ids = np.unique(np.concatenate([vis[vis != R.VIS_NONE], big]))
    assert ids.size > 1000
    rec = r.debug_read(R.DEBUG_TRI_RECORDS | R.DEBUG_AS_DRAWN, np.uint32).reshape(-1, 16)[ids]
    flags, orec = O.setup(sc, cam, opts.cull_mode, W, H)
    assert flags[ids].all()
    np.testing.assert_array_equal(np.ascontiguousarray(rec[:, [0, 1, 2, 3, 4, 5, 6, 9, 8, 7, 10, 11]]),
                                  np.ascontiguousarray(orec[ids]).view(np.uint32))
    tri = indices(sc)[ids]
    np.testing.assert_array_equal(np.sort(rec[:, 12:15], axis=1), np.sort(tri, axis=1))
    mesh = np.repeat(np.arange(len(sc.meshes)), [m.num_triangles for m in sc.meshes])[ids]
    np.testing.assert_array_equal(rec[:, 15] & 0x7FFFFFFF, mesh + first_mesh)
    both = [O.vertex_transform(sc, cam, W, H, k) for k in range(len(sc.meshes))]
    opos, oattr = (np.concatenate([b[q] for b in both]).astype(np.float32) for q in range(2))
    v = np.unique(tri)
    pos = r.debug_read(R.DEBUG_VERTEX_POS | R.DEBUG_AS_DRAWN, np.uint32).reshape(-1, 4)
    np.testing.assert_array_equal(pos[v], np.ascontiguousarray(opos[v]).view(np.uint32))
    if attributes:
        attr = r.debug_read(R.DEBUG_VERTEX_ATTR | R.DEBUG_AS_DRAWN, np.float32).reshape(-1, 12)[v]
        inv_w = oattr[v, 14:15]
        want = np.concatenate([(oattr[v, :11] * inv_w).astype(np.float32), inv_w], axis=1)
        got = np.ascontiguousarray(attr[:, [0, 1, 3, 4, 5, 6, 7, 8, 9, 10, 11, 2]])
        np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("kind", ["list", "strip", "shuffled"])
@pytest.mark.parametrize("policy", [R.BIN_EXACT, R.BIN_PREVFRAME])
def test_single_frames(kind, policy):
    sc, opts = scene(kind), S.Opts(cull_mode=S.CULL_NONE)
    with R.Renderer(W, H) as r:
        r.add_scene(sc)
        for turn in range(2):
            for cam in CAMERAS:  # each leaves its entries for the next to be taken for
                r.render(cam, opts, policy)
                check(r, sc, cam, opts)


@pytest.mark.parametrize("kind", ["list", "strip", "shuffled"])
def test_views(kind):
    sc, opts = scene(kind), S.Opts(cull_mode=S.CULL_NONE)
    owner = R.Renderer(W, H)
    owner.add_scene(sc)
    rs = [owner] + [owner.view(W, H) for _ in range(13)]
    try:
        for turn in range(3):
            cams = [CAMERAS[(k + turn) % len(CAMERAS)] for k in range(len(rs))]
            R.render_batch([(r, cam, opts, R.BIN_EXACT, 0) for r, cam in zip(rs, cams)])
            for k, (r, cam) in enumerate(zip(rs, cams)):
                check(r, sc, cam, opts, attributes=False, first_mesh=2 * k)
    finally:
        for r in rs[:0:-1]:
            r.close()
        owner.close()


def test_only_what_a_frame_forms_can_be_asked_for():
    with R.Renderer(W, H) as r:
        r.add_scene(scene("list"))
        r.render(CAMERAS[0], S.Opts())
        for which in (R.DEBUG_TRI_ALIVE, R.DEBUG_TILE_COUNTS, R.DEBUG_BIG_LIST, R.DEBUG_TILE_CAPS):
            with pytest.raises(R.RastError, match="unknown debug buffer"):
                r.debug_read(which | R.DEBUG_AS_DRAWN)
