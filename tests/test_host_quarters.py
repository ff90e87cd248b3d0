"""Tiles are resolved in quarters where the launch, all its frames together,
leaves the chip idle.  Host code only."""
import pytest

import rast as R
import scenes as S


@pytest.mark.parametrize("frames,quarters", [
    ([(640, 480, 32)], True),                          # 300 tiles
    ([(640, 480, 32), (512, 384, 32)], True),          # 492
    ([(640, 480, 32), (640, 480, 32)], False),         # 600
    ([(640, 480, 32), (256, 208, 16)], True),          # 300 + 208
    ([(640, 480, 32), (256, 224, 16)], False),         # 300 + 224
    ([(640, 480, 32), (1920, 1080, 16)], False),       # 300 beside 8,160
    ([(64, 64, 32), (640, 480, 8)], False),            # 4 beside 4,800
    ([(320, 256, 16)], False),                         # no tiles of 32 pixels
])
def test_which_launches_take_quarters(host, frames, quarters):
    rs = [R.Renderer(w, h, tile=t) for w, h, t in frames]
    for r in rs:
        r.add_mesh(S.uv_sphere(8, 4, 1.0))
    host.launches.clear()
    R.render_batch([(r, S.Camera(), S.Opts(), R.BIN_EXACT, 0) for r in rs])
    grids = {n: sum(g for m, g, _ in host.launches if m == n) for n in ("k_resolve", "k_resolve_quarters")}
    whole = [-(-w // t) * -(-h // t) for w, h, t in frames]
    parts = sum(n for n, (_, _, t) in zip(whole, frames) if t == 32) if quarters else 0
    assert grids == {"k_resolve": sum(whole) - parts, "k_resolve_quarters": 4 * parts}
    for r in rs:
        r.set_resolve_mode(R.RESOLVE_PERSISTENT)
    host.launches.clear()
    R.render_batch([(r, S.Camera(), S.Opts(), R.BIN_EXACT, 0) for r in rs])
    assert "k_resolve_quarters" not in host.names()
    for r in rs:
        r.close()
