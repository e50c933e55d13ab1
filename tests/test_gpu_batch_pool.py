"""The per-call block that batches keep between calls counts as cached memory,
is given back, and obeys the pool's cap."""
import ctypes

import numpy as np
import pytest

import imresh_amd as im
from helpers import FLT_MIN

pytestmark = pytest.mark.gpu
L = im.lib
BLOCK = 64 << 10   # its smallest size


def _cached():
    b = ctypes.c_uint64()
    im.check(L().imresh_cached_bytes(ctypes.byref(b)))
    return b.value


def test_block_is_counted_released_and_capped():
    x = np.random.default_rng(1).random((4, 4), dtype=np.float32)
    p = im.default_params(n_cycles=1, n_hio_cycles=1, target_error=FLT_MIN)

    def batch():
        out = [x.copy()]
        im.shrink_wrap_batch(out, p)
        im.sync()
        return out[0]

    ref = batch()
    im.check(L().imresh_release_cached())
    assert _cached() == 0
    batch()
    assert _cached() >= BLOCK   # a 4 x 4 class alone takes a few KiB
    try:
        im.check(L().imresh_set_option(2, 0))   # IMRESH_OPT_POOL_MIB
        assert _cached() == 0
        assert np.array_equal(batch(), ref)
        # what was returned last may still have counted as busy: re-apply
        im.sync()
        im.check(L().imresh_set_option(2, 0))
        assert _cached() == 0
        im.check(L().imresh_set_option(2, 1))
        for _ in range(3):
            assert np.array_equal(batch(), ref)
            assert _cached() <= 1 << 20
    finally:
        im.check(L().imresh_set_option(2, 32768))
    im.check(L().imresh_release_cached())
    assert _cached() == 0
