"""Per-operator calls captured in a caller's graph: the pooled scratch buffer
of the captured call stays usable by others, however often the graph is
replayed."""
import ctypes

import numpy as np
import pytest

import imresh_amd as im

pytestmark = pytest.mark.gpu
L = im.lib
RELAXED = 2   # hipStreamCaptureModeRelaxed


def _cached():
    b = ctypes.c_uint64()
    im.check(L().imresh_cached_bytes(ctypes.byref(b)))
    return b.value


def _hip(name, *args):
    # the runtime the library is linked against
    assert getattr(L(), name)(*args) == 0, name


def test_replays_do_not_keep_the_scratch_buffer():
    w, h = 201, 160
    x = np.random.default_rng(4).random((h, w), dtype=np.float32)
    d, e = im.DeviceBuffer.from_array(x), im.DeviceBuffer.from_array(x)
    s = ctypes.c_void_p(im.stream_create())
    graph, run = ctypes.c_void_p(), ctypes.c_void_p()

    def blur(buf):
        im.check(L().imresh_gaussian_blur(buf.ptr, w, h, 2.0, s))

    def eager(buf):
        blur(buf)
        im.sync(s)

    im.check(L().imresh_release_cached())
    eager(d)   # the buffer and the weights exist from here on
    idle = _cached()
    assert idle > 0
    eager(e)
    _hip("hipStreamBeginCapture", s, ctypes.c_int(RELAXED))
    blur(d)
    _hip("hipStreamEndCapture", s, ctypes.byref(graph))
    _hip("hipGraphInstantiate", ctypes.byref(run), graph, None, None, ctypes.c_size_t(0))
    try:
        for _ in range(4):
            _hip("hipGraphLaunch", run, s)
            im.sync(s)
            assert _cached() == idle   # not taken for busy
            eager(e)
            assert np.array_equal(d.download(np.float32, (h, w)), e.download(np.float32, (h, w)))
            assert _cached() == idle   # nor has another one been made
    finally:
        _hip("hipGraphExecDestroy", run)
        _hip("hipGraphDestroy", graph)
        im.stream_destroy(s)
    im.check(L().imresh_release_cached())
    assert _cached() == 0
