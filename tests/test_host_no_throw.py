"""Entry points that find no host memory return RAST_E_OUT_OF_MEMORY, throw
nothing, lose nothing, and the same call succeeds afterwards: every allocation
that a call makes fails once.  Host code only."""
import ctypes as C

import numpy as np
import pytest

import rast as R
import scenes as S

OUT_OF_MEMORY = -3


def every_allocation(host, call, done=None):
    """Runs `call` with its first, second, ... allocation failing, until none does."""
    for k in range(400):
        host.lib.stub_fail_new(k)
        try:
            out = call()
        except R.RastError as e:
            assert f"({OUT_OF_MEMORY})" in str(e), e
            failed = True
        else:
            failed = False
        left = host.lib.stub_fail_left()
        host.lib.stub_fail_new(-1)
        if left >= 0:  # it made fewer allocations than that
            assert not failed
            if done:
                done(out)
            return k
        if not failed and done:
            done(out)
    raise AssertionError("no end")


def mesh():
    m = S.uv_sphere(16, 8, 1.0)
    m.textures = S.noise_maps(16, 3)
    return m


def frames(r):
    for flags in (0, R.FLAG_GRAPH, R.FLAG_NO_SHADE):
        r.render(S.Camera(), S.Opts(), R.BIN_EXACT, flags)
    r.sync()


@pytest.fixture
def r(host):
    with R.Renderer(64, 48) as r:
        r.add_mesh(mesh())
        yield r


def test_renderers_and_views(host, r):
    base = host.used(), host.pinned()
    assert every_allocation(host, lambda: R.Renderer(96, 64), lambda x: x.close()) > 0
    assert every_allocation(host, lambda: r.view(96, 64), lambda x: x.close()) > 0
    assert (host.used(), host.pinned()) == base
    frames(r)


def test_meshes_and_textures(host, r):
    lib, v = R.lib(), mesh()

    def create():
        h = C.c_void_p()
        R.check(lib.rast_mesh_create(r.h, v.verts.ctypes.data, v.verts.shape[0], v.indices.ctypes.data, v.indices.size,
                                     v.topology, v.world.ctypes.data, C.byref(h)), "rast_mesh_create")
        return h

    base = host.used()
    assert every_allocation(host, create, lambda h: R.check(lib.rast_mesh_destroy(h))) > 3

    def texture():
        h, t = C.c_void_p(), np.zeros((8, 8), np.uint32)
        R.check(lib.rast_texture_create(r.h, t.ctypes.data, 8, 8, C.byref(h)), "rast_texture_create")
        return h

    assert every_allocation(host, texture, lambda h: R.check(lib.rast_texture_destroy(h))) > 0
    assert host.used() == base
    frames(r)


@pytest.mark.parametrize("flags", [0, R.FLAG_GRAPH])
def test_first_frames(host, flags):
    r = R.Renderer(64, 48)
    r.add_mesh(mesh())
    assert every_allocation(host, lambda: r.render(S.Camera(), S.Opts(), R.BIN_EXACT, flags)) > 5
    frames(r)
    # another shape of launch, from the state a failed one left
    r.setup_bins(32, 64)
    every_allocation(host, lambda: r.render(S.Camera(), S.Opts(sample_state=1), R.BIN_EXACT, flags))
    frames(r)
    r.close()


def test_batches(host, r):
    views = [r.view(64, 64, tile=t) for t in (8, 16, 32)]

    def batch():
        R.render_batch([(x, S.Camera(), S.Opts(), R.BIN_EXACT, 0) for x in [r] + views])

    assert every_allocation(host, batch) > 10
    batch()
    frames(r)
    for v in views[::-1]:
        v.close()


def test_reads(host, r):
    frames(r)
    for which in range(7):
        every_allocation(host, lambda: r.debug_read(which))
        r.render(S.Camera(), S.Opts())
    every_allocation(host, lambda: r.readback())
    every_allocation(host, lambda: r.stats())
    frames(r)


def test_models(host, r):
    base = host.used()
    assert every_allocation(host, lambda: R.BinModel(r, hidden=16), lambda m: m.close()) > 1
    assert host.used() == base
    m = R.BinModel(r, hidden=16)
    every_allocation(host, lambda: m.attach(r))
    for _ in range(3):
        r.render(S.Camera(), S.Opts(), R.BIN_LEARNED)
    every_allocation(host, lambda: m.record(r))
    every_allocation(host, lambda: m.train(1, batch=64))
    every_allocation(host, lambda: m.forward(np.zeros((9, 8), np.float32)))
    m.close()
    frames(r)


def test_destruction_of_meshes(host, r):
    for _ in range(4):
        r.add_mesh(mesh())
        frames(r)
        h = r.meshes.pop()
        host.lib.stub_fail_new(0)
        R.check(R.lib().rast_mesh_destroy(h), "rast_mesh_destroy")
        host.lib.stub_fail_new(-1)
        frames(r)
