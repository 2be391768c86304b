"""Maps with transposed operands against the oracle: results are the same whole numbers (or floats, element by
element) at the edges of the tiles (extents one below, at and above a multiple of 32 and 64), for one and
several transposed views, for axes before the two of the tile, and for every element size."""
import numpy as np
import pytest

import bohrium_amd as bh
from tests.helpers import run_both


def _input(shape, dtype, seed=3):
    n = int(np.prod(shape))
    r = bh.random.RandomState(seed).random123((n,))
    x = (r % np.uint64(251)).astype(dtype).reshape(shape)
    bh.flush()
    return x


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(256, 256), (255, 257), (320, 321), (32, 2049), (2049, 33), (31, 4096), (65, 1023)])
@pytest.mark.parametrize("dtype", [np.bool_, np.int16, np.float32, np.float64, np.complex128])
def test_transposed_operands(shape, dtype):
    def program():
        x, y = _input(shape, dtype), _input(shape[::-1], dtype, 4)
        out = [y.T.copy(), x.T.copy()]
        if np.dtype(dtype) != np.bool_:
            out += [x + y.T, (x + x) * y.T[::-1, ::-1], y.T[:, ::-1] + y.T]
        return out
    got, want = run_both(program)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)


@pytest.mark.gpu
def test_outer_axes_several_views_and_offsets():
    def program():
        x = _input((5, 96, 130), np.float32)
        z = _input((130, 5, 96), np.float64, 8)
        big = _input((200, 300), np.float64, 9)
        return [x.transpose(0, 2, 1) * 2, z.transpose(1, 0, 2) + x.transpose(0, 2, 1), x.transpose(2, 1, 0) + 1,
                big[3:143, 5:290].T + 1,
                big[::2, ::3].T + big[1::2, 1::3].T]
    got, want = run_both(program)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)


@pytest.mark.gpu
def test_many_matrices_in_one_flush():
    """Twelve transposes of one form run as a batched launch (each its own tiles)."""
    def program():
        xs = [_input((300 + i, 260), np.float32, i) for i in range(12)]
        return [x.T + 1 for x in xs]
    got, want = run_both(program)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)
