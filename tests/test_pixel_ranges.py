"""The pixel range setup rasterizes a small triangle over (edge_reach and
first_pixel in rast_kernels.hip, restated in float32) holds every pixel of the
reference's range that passes the three evaluated edge tests, for both
windings: random triangles, needles whose corners are nearly collinear at the
coordinates' resolution, and corners on pixel centres, anywhere on a 16K
screen.  A range planted one pixel short fails."""
import numpy as np
import pytest

f = np.float32
U = 2.0 ** -24


def triangles(kind, n, rng):
    """n triangles' corners, (n, 3) float32 x and y, extents up to about 6 pixels."""
    base = rng.choice([3.0, 60.0, 1000.0, 3900.0, 16000.0], n)[:, None] + rng.uniform(0, 8, (n, 1))
    basey = rng.choice([3.0, 500.0, 2100.0, 16000.0], n)[:, None] + rng.uniform(0, 8, (n, 1))
    if kind == "random":
        ext = 2.0 ** rng.uniform(-6, 2.5, (n, 1))
        x, y = base + rng.uniform(-1, 1, (n, 3)) * ext, basey + rng.uniform(-1, 1, (n, 3)) * ext
    elif kind == "needle":
        t = rng.uniform(-1, 1, (n, 3)) * 2.5
        a = rng.uniform(0, 2 * np.pi, (n, 1))
        a = np.where(rng.random((n, 1)) < 0.3, np.round(a / (np.pi / 4)) * (np.pi / 4), a)
        off = rng.integers(-3, 4, (n, 3)) * 2.0 ** rng.integers(-24, -8, (n, 1))
        x, y = base + t * np.cos(a) - off * np.sin(a), basey + t * np.sin(a) + off * np.cos(a)
    else:  # corners on pixel centres or a few units in the last place beside them
        x = np.floor(base) + rng.integers(-3, 4, (n, 3))
        y = np.floor(basey) + rng.integers(-3, 4, (n, 3))
        x, y = x.astype(f), y.astype(f)
        for _ in range(2):
            d = rng.integers(-1, 2, (n, 3))
            x = np.where(d > 0, np.nextafter(x, f(1e9)), np.where(d < 0, np.nextafter(x, f(-1e9)), x))
            d = rng.integers(-1, 2, (n, 3))
            y = np.where(d > 0, np.nextafter(y, f(1e9)), np.where(d < 0, np.nextafter(y, f(-1e9)), y))
    return x.astype(f), y.astype(f)


def ranges(x, y, area, reach_scale):
    w, h = x.max(1) - x.min(1), y.max(1) - y.min(1)
    with np.errstate(divide="ignore", over="ignore", invalid="ignore"):
        # the hardware reciprocal is within 1 ulp: the smaller neighbour is the harder case
        rcp = np.nextafter(f(1) / area, f(0))
        reach = f(34.0 / 16777216.0) * np.maximum(np.maximum(w, h), f(2)) * ((w + f(2)) * (h + f(2))) * rcp
    out = []
    for c in (x, y):
        mn = c.min(1)
        lo = np.maximum(np.trunc(mn).astype(np.int64) - 1, 0)
        v = mn - (f(reach_scale) * reach + np.abs(mn) * f(4.0 / 16777216.0))
        out.append((lo, np.ceil(np.fmax(v, lo.astype(f))).astype(np.int64)))
    return out


def uncovered(kind, n, seed, reach_scale=1.0, shift=0):
    """Pixels of the reference's range that pass the edge tests and are left out."""
    rng = np.random.default_rng(seed)
    x, y = triangles(kind, n, rng)
    cr = (x[:, 0] - x[:, 1]) * (y[:, 0] - y[:, 2]) - (y[:, 0] - y[:, 1]) * (x[:, 0] - x[:, 2])
    keep = (cr != 0) & np.isfinite(cr)
    x, y, area = x[keep], y[keep], np.abs(cr[keep])
    (lx, tx), (ly, ty) = ranges(x, y, area, reach_scale)
    tx = tx + shift
    hx, hy = np.trunc(x.max(1)).astype(np.int64) + 1, np.trunc(y.max(1)).astype(np.int64) + 1
    assert np.all(tx >= lx) and np.all(ty >= ly)
    missed = dropped = 0
    nx, ny = int((hx - lx).max()), int((hy - ly).max())
    ex = [x[:, (j + 1) % 3] - x[:, j] for j in range(3)]
    ey = [y[:, (j + 1) % 3] - y[:, j] for j in range(3)]
    for j in range(ny):
        for i in range(nx):
            px, py = lx + i, ly + j
            out = (px < tx) | (py < ty)
            there = (px < hx) & (py < hy) & out
            inside = there.copy()
            for k in range(3):
                e = (px.astype(f) - x[:, k]) * ey[k] - (py.astype(f) - y[:, k]) * ex[k]
                inside &= e >= 0
            missed += int(inside.sum())
            dropped += int(there.sum())
    return missed, dropped


@pytest.mark.parametrize("kind", ["random", "needle", "centres"])
@pytest.mark.parametrize("seed", [1, 2, 3])
def test_every_covered_pixel_is_in_the_range(kind, seed):
    missed, dropped = uncovered(kind, 120000, seed)
    assert missed == 0
    if kind == "random":
        # every range starts a column and a row before its corners: at least 3 pixels
        assert dropped > 2 * 120000


def test_a_range_one_pixel_short_loses_pixels():
    assert uncovered("centres", 120000, 1, 0.0, shift=1)[0] > 0
