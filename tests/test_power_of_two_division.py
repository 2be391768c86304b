"""Division by a constant power of two is a multiplication: the same bits as the division over the whole range of
the types (infinities, NaN, zeros, subnormal operands and results, both signs), and a plan cached for one divisor is not
used for a divisor that needs the other form."""
import numpy as np
import pytest

import bohrium_amd as bh

pytestmark = pytest.mark.gpu


def _values(dtype):
    f = np.finfo(dtype)
    r = np.random.RandomState(3)
    e = r.randint(f.minexp - f.nmant, f.maxexp, 60000)
    x = np.ldexp(r.uniform(0.5, 1, 60000).astype(dtype), e).astype(dtype) * r.choice([-1, 1], 60000).astype(dtype)
    return np.concatenate([x, np.array([0.0, -0.0, np.inf, -np.inf, np.nan, f.max, f.min, f.tiny, -f.tiny, f.smallest_subnormal], dtype)])


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_same_bits(dtype):
    f = np.finfo(dtype)
    h = _values(dtype)
    x = bh.array(h)
    exps = [0, 1, -1, 2, 10, -24, 64, -64, 100, f.maxexp - 2, f.maxexp - 1, f.minexp, f.minexp + 1]
    for k in exps:
        for sign in (1.0, -1.0):
            d = dtype(np.ldexp(sign, k))
            with np.errstate(all="ignore"):
                want = h / d
            got = (x / d).asnumpy()
            np.testing.assert_array_equal(got.view("u%d" % h.itemsize)[~np.isnan(want)],
                                          want.view("u%d" % h.itemsize)[~np.isnan(want)], err_msg=str(k))
            assert np.isnan(got[np.isnan(want)]).all()


def test_cached_plans_keep_the_forms_apart():
    h = np.random.RandomState(4).uniform(-5, 5, 1000)
    x = bh.array(h)
    for d in (4.0, 3.0, 8.0, 0.1, 2.0 ** -3, 7.0, 2.0 ** 64, 4.0):
        np.testing.assert_array_equal((x / d).asnumpy(), h / d)
