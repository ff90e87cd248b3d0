"""Which way frames are binned after one that left many entries beyond its
queue regions: by two passes, at once where its lists were full, and back in
one pass after enough frames that would fit.  Host code only, without a GPU."""
import pytest

import rast as R
import scenes as S

MANY, FEW = 2_000_000, 100
TWO_PASS, PLACED = {"k_place", "k_fill"}, {"k_fallback_alloc", "k_fallback_fill"}


@pytest.fixture
def renderer(host):
    with R.Renderer(320, 200, tile=16) as r:
        r.add_scene(S.Scene([S.uv_sphere(48, 24, 1.0)]))
        yield r


def render(host, r, policy=R.BIN_EXACT, sync=True, **left):
    """One frame, whose counters end as given; the kernels it launched."""
    host.launches.clear()
    done = []

    def end(name):
        if name == "k_shade":
            full = dict(storage_overflow=0, ovf_entries=0, pool_used=0, past_fixed=0, past_spill=0, spilled=0)
            if not done:  # drawn again, it is as it should be
                full.update(left)
            host.counters(**full)
            done.append(name)

    host.on_launch = end
    r.render(S.Camera(), S.Opts(), policy)
    if sync:
        r.sync()
    host.on_launch = None
    return host.names()


def test_a_full_list_goes_to_two_passes_at_once(host, renderer):
    first = render(host, renderer, storage_overflow=1, ovf_entries=MANY, past_fixed=MANY, pool_used=MANY)
    again = first[first.index("k_shade") + 1:]  # the frame drawn again
    assert not TWO_PASS & set(first[:first.index("k_shade")])
    assert TWO_PASS <= set(again)
    assert again.count("k_shade") == 1


def test_the_lists_of_a_frame_that_takes_two_passes_do_not_grow(host, renderer):
    render(host, renderer)
    before = host.used()
    render(host, renderer, storage_overflow=1, ovf_entries=MANY, past_fixed=MANY, pool_used=MANY)
    assert host.used() == before


@pytest.mark.parametrize("sync", [True, False])
def test_two_passes_end_after_frames_that_fit(host, renderer, sync):
    assert not TWO_PASS & set(render(host, renderer, sync=sync, ovf_entries=MANY, past_fixed=MANY))
    routes = [bool(TWO_PASS & set(render(host, renderer, sync=sync, past_fixed=FEW))) for _ in range(40)]
    n = routes.index(False)
    assert routes[0] and 8 <= n <= 32 and not any(routes[n:])
    # one that does not fit starts them again, and so does one among them
    render(host, renderer, sync=sync, past_fixed=MANY)
    routes = [bool(TWO_PASS & set(render(host, renderer, sync=sync, past_fixed=MANY if k == 5 else FEW)))
              for k in range(40)]
    assert routes.index(False) == n + 6


@pytest.mark.parametrize("change", ["resize", "tuning", "bins", "scene"])
def test_a_change_of_the_frame_forgets_them(host, renderer, change):
    render(host, renderer, past_fixed=MANY)
    if change == "resize":
        R.check(R.lib().rast_resize(renderer.h, 256, 256))
    elif change == "tuning":
        renderer.set_tuning(0, 16)
    elif change == "bins":
        renderer.setup_bins(32, 64)
    else:
        renderer.add_mesh(S.uv_sphere(8, 4, 1.0))
    assert not TWO_PASS & set(render(host, renderer))


def test_spill_regions_give_way_to_placing_passes_and_come_back(host, renderer):
    renderer.set_queue_depth(1.0, 0)
    P = R.BIN_PREVFRAME
    render(host, renderer, P)
    assert not PLACED & set(render(host, renderer, P))
    names = render(host, renderer, P, storage_overflow=1, ovf_entries=MANY, spilled=FEW, past_spill=MANY)
    k = names.index("k_shade")
    assert not PLACED & set(names[:k]) and PLACED <= set(names[k:])
    routes = [bool(PLACED & set(render(host, renderer, P, past_spill=FEW))) for _ in range(40)]
    n = routes.index(False)
    assert routes[0] and 8 <= n <= 32 and not any(routes[n:])


def test_frames_that_measure_nothing_change_nothing(host, renderer):
    none = 0xFFFFFFFF
    render(host, renderer, past_fixed=none, past_spill=none)
    assert not TWO_PASS & set(render(host, renderer, past_fixed=none))
    render(host, renderer, past_fixed=MANY)
    for _ in range(40):
        assert TWO_PASS <= set(render(host, renderer, past_fixed=none))
