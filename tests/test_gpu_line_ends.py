"""What lies past the end of a Bluestein line (the next row in memory, and the
transform's own values beyond the line) stays out of the line, also when it is
not finite."""
import numpy as np
import pytest

import imresh_amd as im
from helpers import FLT_MIN

pytestmark = pytest.mark.gpu
B = im.DeviceBuffer
L = im.lib


# one width per convolution length and rows per workgroup: 64, 512, 1024, 4096, 8192, 16384
@pytest.mark.parametrize("w", [20, 150, 300, 1373, 3000, 5000])
def test_row_that_overflows_leaves_the_rows_above_it(w):
    # The modulus alternates down the columns: their inverse transform is 0
    # except in row 128, where 256 values of 1.6e36 sum past the largest float
    # (128 of them do not).
    M = np.repeat(np.where(np.arange(256) % 2, -1.6e36, 1.6e36).astype(np.float32)[:, None], w, 1)
    p = im.default_params(n_cycles=1, target_error=FLT_MIN, n_hio_cycles=1)
    g = im.debug_cycle_mask(M, 0, p)[0]
    assert not np.isfinite(g[128]).any()
    assert np.array_equal(np.delete(g, 128, 0), np.zeros((255, w), np.complex64))


# convolutions of 64, 1024 and 4096 points
@pytest.mark.parametrize("n", [20, 300, 1100])
def test_overflow_beyond_the_line_stays_there(n):
    # Position n + n/2 of the convolution lies past the line: this column adds
    # up to 3.6e38 there and stays below 3.3e38 in the line, so only what has to
    # be left out overflows, between the transform and its inverse.
    j, p = np.arange(n), n // 2
    a = np.exp(-1j * np.pi * (j * j % (2 * n)) / n)
    ahead = np.exp(-1j * np.pi * ((n + p - j) ** 2 % (2 * n)) / n)
    x = 3.6e38 / (n - 1 - p) * np.conj(a) * ahead * np.where(j > p, 1.0, -0.3)
    # gPrev = g' and a vanishing beta: the constraint changes nothing
    d, q = (B.from_array(x.astype(np.complex64).reshape(n, 1)) for _ in range(2))
    mask, M = B.from_array(np.zeros((n, 1), np.uint8)), B.from_array(np.ones((n, 1), np.float32))
    im.check(L().imresh_hio_iterations(d.ptr, q.ptr, mask.ptr, M.ptr, 1, n, np.float32(1e-30), 1, None))
    assert np.isfinite(d.download(np.complex64, (n, 1)).view(np.float32)).all()
