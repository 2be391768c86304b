"""Synced arrays reach the host: many small ones of one flush together (more than one launch takes, sizes around
the 16-byte pieces and the 64 KiB limit, more bytes than the staging memory holds), beside large ones, and with
the index error of the same flush."""
import numpy as np
import pytest

import bohrium_amd as bh
from bohrium_amd import _bh_api as api

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 15, 16, 17, 31, 33, 255, 4095, 4097, 65535, 65536, 65537, 200001]


def _expect(n, k):
    return ((np.arange(n) + k) % 251).astype(np.uint8)


@pytest.mark.parametrize("copies", [1, 7, 40])
def test_sizes(copies):
    arrays = [(n, k, ((bh.arange(n) + k) % 251).astype(np.uint8)) for k in range(copies) for n in SIZES]
    got = bh.asnumpy_many([a for _, _, a in arrays])
    for (n, k, _), g in zip(arrays, got):
        np.testing.assert_array_equal(g, _expect(n, k))
    # later writes on the device reach the host again
    for n, k, a in arrays[:len(SIZES)]:
        a += np.uint8(1)
        np.testing.assert_array_equal(a.asnumpy(), _expect(n, k) + 1)


def test_index_error_of_the_flush_is_raised_once():
    x = bh.arange(100) * 1.0
    y = bh.take(x, np.array([1, 2, 100]))
    with pytest.raises(api.BohriumError, match="out of bounds"):
        y.asnumpy()
    assert float(x.sum()) == 4950.0
    np.testing.assert_array_equal(bh.take(x, np.array([99, 0])).asnumpy(), [99.0, 0.0])


def test_a_condition_ends_a_repeat():
    a = bh.zeros((1000,))

    def body():
        a[...] = a + 1
        return a.max() < 5
    bh.do_while(body, 100)
    np.testing.assert_array_equal(a.asnumpy(), np.full(1000, 5.0))
