"""The scan skeleton's tiles against the oracle for every tile size (scan_items): lengths one below, at and above
a run, a wave's row, a tile and several tiles; neighbouring elements per thread for contiguous arrays and one for
strided ones; products; types of 1 to 16 bytes; infinities and NaN."""
import numpy as np
import pytest

import bohrium_amd as bh
from tests.helpers import run_both

LENGTHS = [2, 63, 257, 1023, 1025, 2047, 2048, 4097, 16383, 16385, 70001]


@pytest.fixture(params=[4, 8, 16, 32, 64])
def items(request):
    bh.message("autotune: off")
    bh.message("codegen: scan_items=%d" % request.param)
    yield request.param
    bh.message("codegen: scan_items=8")
    bh.message("autotune: on")


@pytest.mark.gpu
@pytest.mark.parametrize("n", LENGTHS)
def test_counts_and_sums(items, n):
    def program():
        r = bh.random.RandomState(n).random123((2 * n,)) % np.uint64(1000)
        x = (r.astype(np.float64) * 0.125 - 60.0).astype(np.float32)
        i, w = r.astype(np.int64), r.astype(np.float64) * 0.125 - 60.0
        z = (w * 1j + 1.0).astype(np.complex128)
        bh.flush()
        return [(x[:n] > 0).astype(np.int64).cumsum(), (x[n:] > 0).astype(np.int64).cumsum(), i[:n].cumsum(),
                w[1:n].cumsum(), i[::2].cumsum(), w[::-1].cumsum(), z[:n].cumsum(), bh.take(i, i % n)[:n].cumsum()]
    got, want = run_both(program)
    for k, (g, w) in enumerate(zip(got, want)):
        # (multiples of 1/8 below 2^24: the float sums are exact in any order)
        np.testing.assert_array_equal(g, w, err_msg=str(k))


@pytest.mark.gpu
def test_products_and_special_values(items):
    def program():
        r = bh.random.RandomState(1).random123((5000,))
        p = ((r % np.uint64(2)).astype(np.float64) * 2.0 - 1.0)
        u = (r % np.uint64(7)).astype(np.uint64)
        bh.flush()
        return [p.cumprod(), (u + np.uint64(1)).cumprod()]
    got, want = run_both(program)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)
    h = np.ones(9000)
    h[3000], h[6000] = np.inf, np.nan
    s = bh.array(h).cumsum().asnumpy()
    np.testing.assert_array_equal(s, np.cumsum(h))
