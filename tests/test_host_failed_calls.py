"""A call that fails leaves nothing behind: the calls after it are not told of
its error.  Host code only, over the stand-in runtime."""
import numpy as np
import pytest

import rast as R
import scenes as S


@pytest.fixture
def renderer(host):
    with R.Renderer(64, 48) as r:
        r.add_mesh(S.uv_sphere(16, 8, 1.0))
        r.render(S.Camera(), S.Opts())
        yield r


def no_room(host, call):
    host.limit(0)
    with pytest.raises(R.RastError):
        call()
    host.limit(None)


def frames(r):
    for flags in (0, R.FLAG_GRAPH):
        r.render(S.Camera(), S.Opts(), R.BIN_EXACT, flags)
    R.render_batch([(r, S.Camera(), S.Opts(), R.BIN_EXACT, 0)])
    r.sync()


@pytest.mark.parametrize("what", ["mesh", "texture", "resize", "renderer", "model", "forward"])
def test_frames_after_a_call_without_memory(host, renderer, what):
    r = renderer
    if what == "mesh":
        no_room(host, lambda: r.add_mesh(S.uv_sphere(512, 256, 1.0)))
    elif what == "texture":
        no_room(host, lambda: r.texture(np.zeros((512, 512), np.uint32)))
    elif what == "resize":
        no_room(host, lambda: R.check(R.lib().rast_resize(r.h, 4096, 4096)))
        R.check(R.lib().rast_resize(r.h, 64, 48))
    elif what == "renderer":
        no_room(host, lambda: R.Renderer(512, 512))
    elif what == "model":
        no_room(host, lambda: R.BinModel(r))
    else:
        m = R.BinModel(r, hidden=16)
        no_room(host, lambda: m.forward(np.zeros((100, 8), np.float32)))
        m.close()
    frames(r)


def test_frames_after_a_refused_debug_read(renderer):
    R.check(R.lib().rast_resize(renderer.h, 1024, 1024))
    with pytest.raises(R.RastError):  # more tiles than the last frame had
        renderer.debug_read(R.DEBUG_TILE_COUNTS)
    frames(renderer)


@pytest.mark.parametrize("room", [0, 80 << 20, 150 << 20, 210 << 20])  # none, or vis, depth, colours
@pytest.mark.parametrize("read", [False, True])
def test_a_resize_without_memory_leaves_no_frame(host, renderer, room, read):
    """Its buffers may be gone: nothing draws into them or copies from them."""
    r = renderer
    if read:
        r.readback()
    host.limit(room)
    with pytest.raises(R.RastError):
        R.check(R.lib().rast_resize(r.h, 4096, 4096))
    r.width = r.height = 4096
    host.launches.clear()
    for call in (r.readback, lambda: r.render(S.Camera(), S.Opts()), r.readback,
                 lambda: r.draw_texture(np.zeros((4, 4), np.uint32)),
                 lambda: R.render_batch([(r, S.Camera(), S.Opts(), R.BIN_EXACT, 0)]),
                 lambda: R.check(R.lib().rast_frame_buffers(r.h, None, None, None))):
        with pytest.raises(R.RastError):
            call()
    assert host.names() == []
    host.limit(None)
    frames(r)
