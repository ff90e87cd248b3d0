"""entries_in_view in rast_kernels.hip, restated in float32: where it finds a
vertex chunk's reach out of view, box_outside culls every box inside that
reach (the setup pass then reads none of the chunk's positions)."""
import numpy as np
import pytest

from test_box_cull import box_outside, f, wvp_of


@pytest.mark.parametrize("seed", [5, 6])
def test_every_box_in_a_culled_reach_is_culled(seed):
    rng = np.random.default_rng(seed)
    culled = edge = 0
    for _ in range(2500):
        m = wvp_of(rng)
        n = int(rng.integers(1, 5))
        c = rng.uniform(-60, 60, 3) + rng.normal(0, 2, (n, 3))
        h = 2.0 ** rng.uniform(-12, 4, (n, 3))
        if rng.uniform() < 0.5:  # boxes close to the left plane: a point on it, moved out by a few units
            d = m[:, 0].astype(np.float64) + m[:, 3]
            p = rng.uniform(-20, 20, 3)
            p -= d[:3] * (p @ d[:3] + d[3]) / (d[:3] @ d[:3])
            out = -d[:3] / np.linalg.norm(d[:3])
            h = 2.0 ** rng.uniform(-24, -18, (n, 3))
            c = p + out * np.linalg.norm(p) * 2.0 ** -23 * rng.uniform(0, 200, (n, 1))
        lo, hi = (c - h).astype(f), (c + h).astype(f)
        ulo, uhi = lo.min(0), hi.max(0)
        if box_outside(m, ulo, uhi, 2.0):
            culled += 1
            assert all(box_outside(m, lo[k], hi[k]) for k in range(n))
        edge += box_outside(m, ulo, uhi) != 0 and not box_outside(m, ulo, uhi, 2.0)
    assert culled > 300 and edge > 0
