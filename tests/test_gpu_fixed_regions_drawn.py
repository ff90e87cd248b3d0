"""The fixed-region tests over triangles that face the camera: theirs are binned
and counted, but face away and draw nothing."""
import numpy as np
import pytest

import rast as R
import test_gpu_fixed_regions as T
from scene_util import turned

pytestmark = pytest.mark.gpu


@pytest.fixture
def drawn(monkeypatch):
    plain, check = T.pixel_triangles, T.check
    covered = []

    def checked(r, *args):
        covered.append(int(np.count_nonzero(r.readback()[0] != R.VIS_NONE)))
        return check(r, *args)

    monkeypatch.setattr(T, "pixel_triangles", lambda *args: turned(plain(*args)))
    monkeypatch.setattr(T, "check", checked)
    yield
    assert covered and min(covered) > 30


@pytest.mark.parametrize("tile", [8, 16, 32])
@pytest.mark.parametrize("tiles_wide", [1, 16, 17])
def test_block_rectangles(drawn, tile, tiles_wide):
    T.test_block_rectangles(tile, tiles_wide)


@pytest.mark.parametrize("n", [1500, 9000])
def test_overflowing_regions(drawn, n):
    T.test_overflowing_regions_and_the_two_pass_frames_after_them(n)
