"""The pinned slots that readbacks pass through are shared by a device's
renderers: a bounded number is kept, whatever the number of renderers and
threads, and none after the last renderer.  Host code only."""
import threading

import pytest

import rast as R
import scenes as S

MB = 1 << 20


def made(n, width=2048, height=1100):
    rs = [R.Renderer(width, height) for _ in range(n)]
    for r in rs:
        r.add_mesh(S.uv_sphere(8, 4, 1.0))
        r.render(S.Camera(), S.Opts())
    return rs


def close(rs):
    for r in rs:
        r.close()


def test_many_renderers_share_them(host):
    base = host.pinned()
    rs = made(24, 1024, 512) + made(4)
    without = host.pinned()
    for r in rs:
        for plane in r.readback():
            assert plane.shape == (r.height, r.width)
    assert host.pinned() - without < 17 * MB  # one set of two slots of 8 MB
    close(rs)
    assert host.pinned() == base


def test_a_larger_frame_makes_them_longer_once(host):
    rs = made(1, 512, 512) + made(1)
    rs[0].readback()
    small = host.pinned()
    rs[1].readback()
    large = host.pinned()
    assert large > small + 10 * MB
    rs[0].readback()
    rs[1].readback()
    assert host.pinned() == large
    close(rs)


def test_threads(host):
    rs = made(8)
    without = host.pinned()
    errors = []

    def work(r):
        try:
            for _ in range(5):
                r.readback()
        except Exception as e:  # noqa: BLE001 (reported below)
            errors.append(e)

    ts = [threading.Thread(target=work, args=(r,)) for r in rs]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors
    assert host.pinned() - without < 34 * MB  # two sets
    base = without
    close(rs)
    assert host.pinned() < base


def test_slots_of_a_failed_copy_are_not_kept(host):
    rs = made(1)
    without = host.pinned()
    rs[0].readback()
    host.lib.stub_lose_copies(1)
    with pytest.raises(R.RastError, match="ended early"):
        rs[0].readback()
    host.lib.stub_lose_copies(0)
    assert host.pinned() == without
    rs[0].readback()
    close(rs)


def test_the_last_renderer_gives_them_back(host):
    base, mem = host.pinned(), host.used()
    for _ in range(3):
        rs = made(2)
        rs[0].readback()
        rs[0].close()
        assert host.pinned() > base + 10 * MB  # still for the other one
        rs[1].readback()
        rs[1].close()
        assert host.pinned() == base and host.used() == mem
