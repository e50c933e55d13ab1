"""The photon sum of imresh_poisson_modulus either side of its lanes' whole
batches of 16 loads (65536 lanes): every sample depends on the sum's bits."""
import numpy as np
import pytest

import imresh_amd as im
import oracle

pytestmark = pytest.mark.gpu


# 16 L - 1 (the last lane has 15), 16 L, 16 L + 5, 33 L and a part
@pytest.mark.parametrize("w,h", [(1025, 1023), (1024, 1024), (1329, 789), (2111, 1031)])
def test_sum_order_at_batch_edges(w, h):
    m = np.random.default_rng(w).random((h, w), dtype=np.float32)
    d = im.DeviceBuffer.from_array(m)
    im.check(im.lib().imresh_poisson_modulus(d.ptr, w, h, 1e9, 5, None))
    assert np.array_equal(d.download(np.float32, (h, w)), oracle.poisson_modulus(m, 1e9, 5))
