"""The kernels' own bounds (rast_bounds.h, compiled for the host) under the tests
that hold them against what the kernels evaluate: boxes out of view, reaches of
vertex chunks, pixel ranges; and the face test without a square root against the
normalized one."""
import ctypes as C

import numpy as np
import pytest

import test_box_cull
import test_chunk_cull
import test_pixel_ranges

f = np.float32


@pytest.fixture
def bounds(host_library):
    lib = C.CDLL(host_library)

    def call(name, n, *args):
        conv = [a if isinstance(a, C._SimpleCData) else np.ascontiguousarray(a) for a in args]
        getattr(lib, name)(C.c_size_t(n), *[a if isinstance(a, C._SimpleCData) else C.c_void_p(a.ctypes.data) for a in conv])
        return conv[-1]

    return call


@pytest.fixture
def box(bounds, monkeypatch):
    def outside(m, lo, hi, scale=1.0):
        return int(bounds("bounds_box", 1, np.asarray(m, f), np.asarray(lo, f), np.asarray(hi, f), C.c_float(scale),
                          np.zeros(1, np.uint32))[0])

    restated = test_box_cull.box_outside
    monkeypatch.setattr(test_box_cull, "box_outside", outside)
    monkeypatch.setattr(test_chunk_cull, "box_outside", outside)
    return outside, restated


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_boxes(box, seed):
    test_box_cull.test_a_culled_box_has_every_point_beyond_one_plane(seed)


def test_boxes_on_a_plane(box):
    test_box_cull.test_boxes_on_a_plane_stay_unless_the_margins_are_turned_round()


def test_unbounded_boxes(box):
    test_box_cull.test_boxes_that_are_not_finite_or_reach_the_camera_plane_stay()


@pytest.mark.parametrize("seed", [5, 6])
def test_reaches(box, seed):
    test_chunk_cull.test_every_box_in_a_culled_reach_is_culled(seed)


def test_reaches_of_chunks_that_no_triangle_uses(box):
    # their words stay all ones, which read back as NaN: never out of view
    m = test_box_cull.wvp_of(np.random.default_rng(3))
    assert box[0](m, [np.nan] * 3, [np.nan] * 3, 2.0) == 0


@pytest.mark.parametrize("scale", [1.0, 2.0])
def test_the_restatement_agrees(box, scale):
    kernel, restated = box
    rng = np.random.default_rng(8)
    n = 0
    for _ in range(3000):
        m = test_box_cull.wvp_of(rng)
        c, h = rng.uniform(-60, 60, 3), 2.0 ** rng.uniform(-20, 4, 3)
        lo, hi = (c - h).astype(f), (c + h).astype(f)
        assert kernel(m, lo, hi, scale) == restated(m, lo, hi, scale)
        n += kernel(m, lo, hi, scale) != 0
    assert n > 1000


@pytest.fixture
def pixel_ranges(bounds, monkeypatch):
    def ranges(x, y, area, reach_scale):
        w, h = (x.max(1) - x.min(1)).astype(f), (y.max(1) - y.min(1)).astype(f)
        n = len(area)
        reach = bounds("bounds_reach", n, w, h, area.astype(f), np.zeros(n, f)) * f(reach_scale)
        out = []
        for c in (x, y):
            mn = c.min(1)
            lo = np.maximum(np.trunc(mn).astype(np.int64) - 1, 0)
            first = bounds("bounds_first", n, mn, reach, lo.astype(np.int32), np.zeros(n, np.int32))
            out.append((lo, first.astype(np.int64)))
        return out

    monkeypatch.setattr(test_pixel_ranges, "ranges", ranges)
    return ranges


@pytest.mark.parametrize("kind", ["random", "needle", "centres"])
@pytest.mark.parametrize("seed", [1, 2, 3])
def test_pixels(pixel_ranges, kind, seed):
    test_pixel_ranges.test_every_covered_pixel_is_in_the_range(kind, seed)


def test_first_pixels_of_extreme_corners(bounds):
    big = np.array([np.nan, -np.inf, -1e30, 1e30, np.inf, 0.0, -0.0, 5.0, 5.0, 5.0, 5.0], f)
    reach = np.array([0, 0, 0, 0, 0, 0, 0, 0, 1e-3, np.inf, np.nan], f)
    lo = np.full(big.size, 3, np.int32)
    got = bounds("bounds_first", big.size, big, reach, lo, np.zeros(big.size, np.int32))
    assert list(got[[0, 1, 2, 5, 6, 7, 8, 9, 10]]) == [3, 3, 3, 3, 3, 5, 5, 3, 3]


def normalized_faces(c, n, sign):
    """The face test on the normalized normal, in binary32 in the kernel's order."""
    with np.errstate(all="ignore"):
        m = np.sqrt(((n[:, 0] * n[:, 0] + n[:, 1] * n[:, 1]) + n[:, 2] * n[:, 2]).astype(f))
        inv = f(1) / m
        u = np.where((m == 0)[:, None], f(0), n * inv[:, None])
        cv = (c[:, 0] * u[:, 0] + c[:, 1] * u[:, 1]) + c[:, 2] * u[:, 2]
        return ~(cv <= 0) if sign > 0 else ~(cv >= 0)


@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_faces_decide_as_the_normalized_normal(bounds, sign):
    rng = np.random.default_rng(11)
    n = 400000
    c = rng.normal(0, 1, (n, 3))
    c /= np.linalg.norm(c, axis=1, keepdims=True)
    c[: n // 8] = np.round(c[: n // 8])  # along the axes, and zero
    v = rng.normal(0, 1, (n, 3)) * 10.0 ** rng.uniform(-25, 20, (n, 1))
    # half of them across the camera's direction, but for a few units in the last place
    half = slice(n // 2, None)
    p = v[half] - c[half] * (v[half] * c[half]).sum(1, keepdims=True)
    v[half] = p * (1 + 2.0 ** -23 * rng.integers(-6, 7, p.shape))
    with np.errstate(all="ignore"):
        c, v = c.astype(f), v.astype(f)
    v[:64] = rng.choice([0.0, -0.0, np.inf, -np.inf, np.nan, 1e-30, 3e38], (64, 3))
    got = bounds("bounds_faces", n, c, v, C.c_float(sign), np.zeros(n, np.uint8)).astype(bool)
    np.testing.assert_array_equal(got, normalized_faces(c, v, sign))
    assert 0.1 < got.mean() < 0.9
