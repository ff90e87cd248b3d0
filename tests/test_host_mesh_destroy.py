"""Destroying a mesh does no work on the device: its geometry stays for the
last frames' debug buffers until the next frames, or until an allocation needs
the room, after which those buffers are refused.  Host code only."""
import numpy as np
import pytest

import rast as R
import scenes as S

DEBUG = (R.DEBUG_VERTEX_POS, R.DEBUG_VERTEX_ATTR, R.DEBUG_TRI_RECORDS, R.DEBUG_TRI_ALIVE)


def big():
    return S.uv_sphere(512, 256, 1.0)  # 131,841 vertices of 56 bytes


BYTES = 513 * 257 * 56


def render(r):
    r.render(S.Camera(), S.Opts())


def destroy(r, k):
    R.check(R.lib().rast_mesh_destroy(r.meshes.pop(k)), "rast_mesh_destroy")


@pytest.fixture
def drawn(host):
    """An owner and two views that have drawn a small and a big mesh."""
    base = host.used()
    owner = R.Renderer(160, 96)
    owner.add_mesh(S.uv_sphere(8, 4, 1.0))
    owner.add_mesh(big())
    rs = [owner, owner.view(160, 96), owner.view(64, 64)]
    for r in rs:
        render(r)
    host.launches.clear()
    yield host, rs
    for r in rs[::-1]:
        r.close()
    assert host.used() == base


def test_no_work_at_the_destruction(drawn):
    host, rs = drawn
    before, mallocs = host.used(), host.mallocs()
    destroy(rs[0], 1)
    assert host.names() == [] and host.mallocs() == mallocs and host.used() == before
    render(rs[0])
    render(rs[1])
    assert host.used() == before  # the second view's last frame still has it
    render(rs[2])
    assert host.used() <= before - BYTES


def test_debug_buffers_of_the_frames_before(drawn):
    host, rs = drawn
    destroy(rs[0], 1)
    for r in rs:
        for which in DEBUG:
            assert r.debug_read(which).size
        names = host.names()
        assert names.count("k_vertex") == 1 and names.count("k_setup") == 1  # formed once
    render(rs[0])
    for r in rs:  # whole, or of the new frame
        for which in DEBUG:
            r.debug_read(which)


def test_without_frames_it_is_freed_at_once(host):
    with R.Renderer(160, 96) as r:
        r.add_mesh(big())
        before = host.used()
        destroy(r, 0)
        assert host.used() <= before - BYTES


@pytest.mark.parametrize("what", ["mesh", "texture", "frame", "model"])
def test_an_allocation_takes_the_room_back(drawn, what):
    host, rs = drawn
    destroy(rs[0], 1)
    host.limit(BYTES // 2)  # room for it only with the old geometry given back
    if what == "mesh":
        rs[0].add_mesh(S.uv_sphere(512, 200, 1.0))
    elif what == "texture":
        rs[0].texture(np.zeros((1200, 1200), np.uint32))
    elif what == "frame":
        R.check(R.lib().rast_resize(rs[0].h, 640, 480), "rast_resize")
    else:
        m = R.BinModel(rs[0], hidden=16)
        m.forward(np.zeros((150000, 8), np.float32))
        m.close()
    host.limit(None)
    for r in rs:
        for which in DEBUG:
            with pytest.raises(R.RastError, match="scene is gone"):
                r.debug_read(which)
        render(r)
        for which in DEBUG:
            assert r.debug_read(which).size
