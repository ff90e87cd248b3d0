"""Queue storage grows for the tiles' regions only where a frame of the policy
can have them, no further than the scene can fill, and a frame that finds no
memory for it is drawn all the same.  Host code only."""
import numpy as np
import pytest

import rast as R
import scenes as S

BIG = 64  # quads an edge: 8,192 triangles


def frame(host, width, height, tile, policy, scene, frames=1, limit=None, model=False):
    """(bytes of device memory, kernels of the last frame)"""
    base = host.used()
    with R.Renderer(width, height, tile=tile) as r:
        r.add_mesh(scene)
        r.set_queue_depth(1.0, 0)
        m = R.BinModel(r, hidden=16) if model else None
        if m:
            m.attach(r)
        if limit is not None:
            host.limit(limit)
        for _ in range(frames):
            host.launches.clear()
            r.render(S.Camera(), S.Opts(), policy, R.FLAG_NO_SHADE)
            r.sync()
        used, names = host.used() - base, host.names()
        host.limit(None)
        if m:
            m.close()
    return used, names


def per_frame(width, height, tile):
    """Bytes of a frame but for the queues: pixels (20 each) and tiles (nine words)."""
    return 20 * width * height + 36 * -(-width // tile) * -(-height // tile)


FIXED = 60 << 20  # lists, pool, the default queue of 4 MB, a small scene


@pytest.mark.parametrize("policy", [R.BIN_EXACT, R.BIN_PREVFRAME])
@pytest.mark.parametrize("size", [(7680, 4320, 8), (16384, 16384, 16)])
def test_none_where_the_regions_would_be_too_short(host, policy, size):
    used, names = frame(host, *size, policy, S.terrain(BIG), frames=2)
    if policy == R.BIN_EXACT:
        assert "k_place" in names and used < per_frame(*size) + FIXED
    else:  # shorter spill regions are still worth having, within the limit
        assert used < per_frame(*size) + FIXED + (256 << 20)


def test_none_for_learned_capacities(host):
    used, _ = frame(host, 1920, 1080, 8, R.BIN_LEARNED, S.terrain(BIG), frames=3, model=True)
    assert used < per_frame(1920, 1080, 8) + FIXED
    used, names = frame(host, 1920, 1080, 8, R.BIN_LEARNED, S.terrain(BIG))  # without a model: exact
    assert "k_place" not in names and used > per_frame(1920, 1080, 8) + (120 << 20)


@pytest.mark.parametrize("policy", [R.BIN_EXACT, R.BIN_PREVFRAME])
def test_no_more_than_the_scene_can_fill(host, policy):
    small = S.uv_sphere(6, 4, 1.0)
    tris = small.num_triangles
    used, names = frame(host, 3840, 2160, 16, policy, small, frames=2)
    assert not {"k_place", "k_fallback_alloc"} & set(names)
    assert used < per_frame(3840, 2160, 16) + FIXED + 2 * 32400 * tris * 4
    # so few entries a tile that frames of very many tiles have regions too
    used, names = frame(host, 7680, 4320, 8, policy, small, frames=2)
    assert not {"k_place", "k_fallback_alloc"} & set(names)


@pytest.mark.parametrize("policy", [R.BIN_EXACT, R.BIN_PREVFRAME])
def test_a_frame_without_memory_for_it_takes_two_passes(host, policy):
    size = (1920, 1080, 8)
    used, names = frame(host, *size, policy, S.terrain(BIG), frames=3, limit=64 << 20)
    assert names.count("k_resolve") == 1
    assert ("k_place" if policy == R.BIN_EXACT else "k_fallback_alloc") in names
    assert used < per_frame(*size) + FIXED


def test_the_next_size_asks_again(host):
    with R.Renderer(1920, 1080, tile=8) as r:
        r.add_mesh(S.terrain(BIG))
        host.limit(64 << 20)
        r.render(S.Camera(), S.Opts(), R.BIN_EXACT, R.FLAG_NO_SHADE)
        assert "k_place" in host.names()
        host.limit(None)
        mallocs = host.mallocs()
        r.render(S.Camera(), S.Opts(), R.BIN_EXACT, R.FLAG_NO_SHADE)
        assert "k_place" in host.names() and host.mallocs() == mallocs  # not in every frame
        R.check(R.lib().rast_resize(r.h, 1600, 900), "rast_resize")
        r.render(S.Camera(), S.Opts(), R.BIN_EXACT, R.FLAG_NO_SHADE)
        assert "k_place" not in host.names()
