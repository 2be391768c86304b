"""Maps with transposed operands against the oracle: results are the same whole numbers (or floats, element by
element) at the edges of the tiles (extents one below, at and above a multiple of 32 and 64), for one and
several transposed views, for axes before the two of the tile, and for every element size; which maps are
tiled (compile-only)."""
import os
import subprocess
import sys

import numpy as np
import pytest

import bohrium_amd as bh
from tests.helpers import run_both

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
import sys
sys.path.insert(0, %r)
import numpy as np, bohrium_amd as bh
for shape, dtype in %r:
    x = bh.empty(shape, dtype); bh.flush()
    print("PROGRAM", file=sys.stderr, flush=True)
    keep = x.T + x.T if len(shape) == 2 else x.transpose(0, 2, 1) + x.transpose(0, 2, 1)
    bh.flush()
"""
# at and one row below 2^20 elements and 6 MB of a view, and extents below 32
TILED = [((1024, 1024), "float32", True), ((1023, 1024), "float32", False), ((1024, 1024), "int8", True),
         ((1024, 768), "float64", True), ((1023, 768), "float64", False), ((768, 512), "complex128", True),
         ((767, 512), "complex128", False), ((32, 32768), "float32", True), ((31, 40000), "float32", False),
         ((5, 460, 470), "float32", True)]


def test_which_maps_are_tiled():
    r = subprocess.run([sys.executable, "-c", DRIVER % (ROOT, [t[:2] for t in TILED])],
                       env=dict(os.environ, BH_HIP_DRY_RUN="1", BH_HIP_DEBUG="2"), text=True, stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, timeout=600)
    assert r.returncode == 0, r.stdout[-3000:]
    assert ["tl0_[" in part for part in r.stdout.split("PROGRAM")[1:]] == [t[2] for t in TILED]


def _input(shape, dtype, seed=3):
    n = int(np.prod(shape))
    r = bh.random.RandomState(seed).random123((n,))
    x = (r % np.uint64(251)).astype(dtype).reshape(shape)
    bh.flush()
    return x


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(256, 256), (1024, 1024), (1023, 1026), (1088, 1089), (32, 32769), (32769, 33), (31, 34000), (65, 16385)])
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
        x = _input((5, 460, 470), np.float32)
        z = _input((470, 5, 460), np.float64, 8)
        big = _input((1500, 2300), np.float64, 9)
        return [x.transpose(0, 2, 1) * 2, z.transpose(1, 0, 2) + x.transpose(0, 2, 1), x.transpose(2, 1, 0) + 1,
                big[3:1100, 5:2000].T + 1,
                big[::2, ::3].T + big[1::2, 1::3].T]
    got, want = run_both(program)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)


@pytest.mark.gpu
def test_many_matrices_in_one_flush():
    """Twelve transposes of one form run as a batched launch (each its own tiles)."""
    def program():
        xs = [_input((1030 + i, 1025), np.float32, i) for i in range(12)]
        return [x.T + 1 for x in xs]
    got, want = run_both(program)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)
