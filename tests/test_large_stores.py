"""Results of 128 MiB and more are stored past the caches: the values are all there, for every element size,
flat, transposed, in place and scanned, and the next kernel and the host read them."""
import numpy as np
import pytest

import bohrium_amd as bh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.bool_, np.int8, np.int16, np.float32, np.float64, np.complex64])
def test_maps(dtype):
    n = (128 << 20) // np.dtype(dtype).itemsize + 5
    h = (np.arange(n, dtype=np.uint32) % 113).astype(dtype)
    x = bh.array(h)
    y = (x == x) if dtype == np.bool_ else x + x
    bh.flush()
    want = h + h if dtype != np.bool_ else np.ones(n, bool)
    if dtype == np.int8:
        want = (h.astype(np.int16) * 2).astype(np.int8)
    z = y.copy()  # a kernel that reads what was just stored
    bh.flush()
    np.testing.assert_array_equal(y.asnumpy(), want)
    np.testing.assert_array_equal(z.asnumpy(), want)


def test_transposed_scanned_and_in_place():
    r, c = 5001, 6803
    h = (np.arange(r * c) % 1009).astype(np.float32).reshape(r, c)
    x = bh.array(h)
    np.testing.assert_array_equal((x.T + 1).asnumpy(), h.T + 1)
    n = (128 << 20) // 8 + 3
    b = bh.array((np.arange(n) % 3 == 0).astype(np.float32))
    np.testing.assert_array_equal((b > 0).astype(np.int64).cumsum().asnumpy(), np.cumsum(np.arange(n) % 3 == 0))
    x[1:-1, 1:-1] = (x[:-2, 1:-1] + x[2:, 1:-1] + x[1:-1, 2:]) * 0.5
    bh.flush()
    want = h.copy()
    want[1:-1, 1:-1] = (h[:-2, 1:-1] + h[2:, 1:-1] + h[1:-1, 2:]) * np.float32(0.5)
    np.testing.assert_array_equal(x.asnumpy(), want)
