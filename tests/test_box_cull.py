"""box_outside in rast_kernels.hip, restated in float32: a box it culls holds no
point whose evaluated clip position passes the plane the box is beyond, for
boxes beside, behind and across the camera, near the planes, small and large;
and it culls most boxes that are out of view.  With the margins of the wrong
sign, a box placed on a plane is culled although some of its points are not
outside."""
import numpy as np
import pytest

import oracle as O
import scenes as S

f = np.float32
U = f(2.0 ** -24)


def wvp_of(rng):
    d = rng.normal(0, 1, 3)
    d /= np.linalg.norm(d)
    cam = S.Camera(position=tuple(rng.uniform(-40, 40, 3)), forward=tuple(d), fov_deg=float(rng.uniform(20, 120)))
    m = np.asarray(list(O.camera_frame(cam, 640, 480).viewproj), f).reshape(4, 4)  # data[col][row]
    w = S.world_matrix(tuple(rng.uniform(-5, 5, 3)), tuple(rng.uniform(0, 6.28, 3)), float(rng.uniform(0.2, 4)))
    w = np.asarray(w, f).reshape(4, 4)
    return (w.astype(np.float64) @ m.astype(np.float64)).astype(f)  # row vectors of columns: w then m


def clip(m, p):
    """The vertex pass's clip coordinates: (n, 4) float32."""
    return np.stack([((m[0, r] * p[:, 0] + m[1, r] * p[:, 1]).astype(f) + m[2, r] * p[:, 2]).astype(f) + m[3, r]
                     for r in range(4)], 1)


def box_outside(m, lo, hi, scale=1.0):
    """Bit set of the planes the box is beyond (0: not culled)."""
    a = np.maximum(np.abs(lo), np.abs(hi))
    s = [f(np.abs(m[0, r]) * a[0] + np.abs(m[1, r]) * a[1] + np.abs(m[2, r]) * a[2] + np.abs(m[3, r])) for r in range(4)]
    if not all(x < 1e30 for x in s):
        return 0
    k = f(scale)
    ew = k * 16 * U * s[3] + f(1e-30)
    e = [k * 32 * U * (s[r] + s[3]) for r in range(3)]
    c = np.array([[hi[0] if q & 1 else lo[0], hi[1] if q & 2 else lo[1], hi[2] if q & 4 else lo[2]] for q in range(8)], f)
    v = clip(m, c)
    sg = np.where(v[:, 3] < 0, f(-1), f(1))
    w = np.abs(v[:, 3])
    x, y, z = (v[:, r] * sg for r in range(3))
    if not ((v[:, 3] > ew).all() or (v[:, 3] < -ew).all()):
        return 0
    tests = [(x + w < -e[0]), (x - w > e[0]), (y + w < -e[1]), (y - w > e[1]), (z < -e[2]), (z - w > e[2])]
    return sum(1 << i for i, t in enumerate(tests) if t.all())


def outside(m, p):
    """Per plane: which points' evaluated NDC lie beyond it."""
    v = clip(m, p)
    with np.errstate(divide="ignore", invalid="ignore"):
        n = v[:, :3] / v[:, 3:]
    return [n[:, 0] < -1, n[:, 0] > 1, n[:, 1] < -1, n[:, 1] > 1, n[:, 2] < 0, n[:, 2] > 1]


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_a_culled_box_has_every_point_beyond_one_plane(seed):
    rng = np.random.default_rng(seed)
    culled = visible_free = 0
    for _ in range(1500):
        m = wvp_of(rng)
        c, h = rng.uniform(-60, 60, 3), 2.0 ** rng.uniform(-12, 4, 3)
        lo, hi = (c - h).astype(f), (c + h).astype(f)
        p = (rng.uniform(0, 1, (60, 3)) * (hi - lo) + lo).astype(f)
        p = np.clip(np.concatenate([p, np.array([[(lo, hi)[q >> i & 1][i] for i in range(3)] for q in range(8)], f)]), lo, hi)
        out = outside(m, p)
        got = box_outside(m, lo, hi)
        for i in range(6):
            if got >> i & 1:
                assert out[i].all()
        culled += got != 0
        visible_free += any(o.all() for o in out)
    assert culled > 0.8 * visible_free > 500


def test_boxes_on_a_plane_stay_unless_the_margins_are_turned_round():
    # boxes a few units in the last place beyond the left plane of a fixed view
    rng = np.random.default_rng(9)
    wrong = 0
    for _ in range(4000):
        m = wvp_of(rng)
        # a point on the plane x = -w, then a tiny box around it
        d = m[:, 0].astype(np.float64) + m[:, 3]
        p = rng.uniform(-20, 20, 3)
        p -= d[:3] * (p @ d[:3] + d[3]) / (d[:3] @ d[:3])
        n = -d[:3] / np.linalg.norm(d[:3])
        p = p + n * np.linalg.norm(p) * 2.0 ** -23 * rng.uniform(-2, 4)
        lo = p.astype(f)
        hi = np.nextafter(lo, f(1e9))
        pts = np.array([[(lo, hi)[q >> i & 1][i] for i in range(3)] for q in range(8)], f)
        pts = np.concatenate([pts, ((lo + hi) * f(0.5))[None]])
        out = outside(m, pts)
        got = box_outside(m, lo, hi)
        for i in range(6):
            if got >> i & 1:
                assert out[i].all()
        bare = box_outside(m, lo, hi, -1.0)
        wrong += any(bare >> i & 1 and not out[i].all() for i in range(6))
    assert wrong > 0


def test_boxes_that_are_not_finite_or_reach_the_camera_plane_stay():
    rng = np.random.default_rng(4)
    m = wvp_of(rng)
    inf = f(np.inf)
    with np.errstate(invalid="ignore", over="ignore"):
        assert box_outside(m, np.array([-inf] * 3), np.array([inf] * 3)) == 0
        assert box_outside(m, np.array([-1e30] * 3, f), np.array([1e30] * 3, f)) == 0
    big = np.array([200.0] * 3, f)
    assert box_outside(m, -big, big) == 0
