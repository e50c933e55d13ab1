"""Variant numbers that a program may have pinned (an earlier
imresh_autotune's report) stay accepted, and compute the same bits."""
import ctypes

import numpy as np
import pytest

import imresh_amd as im

pytestmark = pytest.mark.gpu
B = im.DeviceBuffer
L = im.lib


# the largest numbers ever reported for lines of 1024 to 8192 points
@pytest.mark.parametrize("w,h,row,col", [(1024, 64, 9, 1), (64, 1024, 3, 9), (2048, 64, 9, 1), (64, 2048, 3, 9),
                                         (4096, 64, 7, 1), (64, 4096, 3, 3), (8192, 64, 7, 1), (64, 8192, 3, 3)])
def test_largest_number_is_accepted(w, h, row, col):
    rng = np.random.default_rng(w + 2 * h)
    g = (rng.random((h, w)) + 1j * rng.random((h, w))).astype(np.complex64)
    mask = (rng.random((h, w)) < 0.5).astype(np.uint8)
    M = rng.random((h, w), dtype=np.float32)
    rv, cv = ctypes.c_int(), ctypes.c_int()

    def run():
        d, q, dm, dM = (B.from_array(a) for a in (g, g, mask, M))
        im.check(L().imresh_hio_iterations(d.ptr, q.ptr, dm.ptr, dM.ptr, w, h, np.float32(0.9), 2, None))
        return d.download(np.float32, (h, 2 * w)), q.download(np.float32, (h, 2 * w))

    im.check(L().imresh_autotune(w, h, None, ctypes.byref(rv), ctypes.byref(cv)))
    tuned, ref = (rv.value, cv.value), run()
    try:
        im.check(L().imresh_set_variants(w, h, row, col))
        im.check(L().imresh_autotune(w, h, None, ctypes.byref(rv), ctypes.byref(cv)))
        assert (rv.value, cv.value) == (row, col)
        for a, b in zip(run(), ref):
            assert np.array_equal(a, b)
    finally:
        im.check(L().imresh_set_variants(w, h, *tuned))
