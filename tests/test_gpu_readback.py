"""A frame's copies to host memory, piece by piece through pinned slots, hold
the bytes of its device buffers: sizes around the chunk and piece edges, ragged
tails, several planes at once, and a destination that is pinned itself."""
import ctypes as C

import numpy as np
import pytest
import torch

import rast as R
import scenes as S

pytestmark = pytest.mark.gpu


class Plane:
    def __init__(self, ptr, shape, kind):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": kind, "data": (ptr, False), "version": 2}


def device_planes(r):
    p = (C.c_void_p(), C.c_void_p(), C.c_void_p())
    R.check(R.lib().rast_frame_buffers(r.h, *(C.byref(q) for q in p)), "rast_frame_buffers")
    return [torch.as_tensor(Plane(q.value, (r.height, r.width), "<i4"), device="cuda") for q in p]


# one pixel; just below and above the staged size; whole chunks; one word past
# a chunk; a whole piece (8 MB) and one row more; several pieces; ragged rows
@pytest.mark.parametrize("width,height", [(1, 1), (511, 256), (512, 256), (513, 257), (16384, 17), (2048, 1024),
                                          (2048, 1025), (4099, 1027), (777, 431)])
def test_readback_bytes(width, height):
    w = S.config1()
    with R.Renderer(width, height) as r:
        r.add_scene(w.scene)
        for frame in range(2):  # the second passes through slots already made
            r.render(w.camera, w.opts)
            planes = device_planes(r)
            # values that depend on the place, so that a misplaced chunk shows
            rng = torch.Generator(device="cuda").manual_seed(width * 7 + frame)
            for t in planes:
                t.copy_(torch.randint(-2**31, 2**31 - 1, t.shape, generator=rng, device="cuda", dtype=torch.int32))
            got = r.readback()
            for t, g in zip(planes, got):
                np.testing.assert_array_equal(t.cpu().numpy().view(np.uint32), g.view(np.uint32))
            only = r.readback(vis=False, depth=False)[2]
            np.testing.assert_array_equal(only, got[2])


def test_readback_into_pinned_and_unaligned_memory():
    w = S.config1()
    with R.Renderer(800, 600) as r:
        r.add_scene(w.scene)
        r.render(w.camera, w.opts)
        want = r.readback()[2]
        pinned = torch.empty((600, 800), dtype=torch.int32, pin_memory=True)
        R.check(R.lib().rast_readback(r.h, None, None, pinned.data_ptr()), "rast_readback")
        np.testing.assert_array_equal(pinned.numpy().view(np.uint32), want)
        raw = np.full(800 * 600 * 4 + 8, 0xA5, np.uint8)
        R.check(R.lib().rast_readback(r.h, None, None, raw.ctypes.data + 4), "rast_readback")
        np.testing.assert_array_equal(raw[4:-4].view(np.uint32).reshape(600, 800), want)
        assert (raw[:4] == 0xA5).all() and (raw[-4:] == 0xA5).all()
