"""Stencils walked by column groups and row bands against the oracle: widths that are 0 to 3 past a multiple of
the column group, heights that end inside a row group and inside a band, 5- and 9-point windows and one that
reaches 3 rows and several columns, beside arrays read at one place, as a map, in place through the twin and
with a maximum; and the plan (what is small keeps the element walk)."""
import os
import subprocess
import sys

import numpy as np
import pytest

import bohrium_amd as bh
from bohrium_amd import workloads
from tests.helpers import run_both

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# interiors (rows - 2, cols - 2) of at least 2^20 elements
SHAPES = [(1026, 1026), (1030, 1027), (1029, 1028), (4099, 261), (263, 4101), (16391, 67)]


def _grid(shape, dtype, seed=2):
    n = int(np.prod(shape))
    r = bh.random.RandomState(seed).random123((n,))
    x = ((r % np.uint64(1 << 20)).astype(np.float64) * (2.0 ** -17) - 4.0).astype(dtype).reshape(shape)
    bh.flush()
    return x


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_jacobi_sweeps(shape, dtype):
    """Sums of five values in program order and one product: the same operations as the oracle's, so the grids
    agree to the last bit; max|new - old| may contract the product and the difference (one rounding of the
    larger value, 8 eps)."""
    def program():
        G = _grid(shape, dtype)
        d = workloads.jacobi_step(G)
        bh.flush()
        d2 = workloads.jacobi_step(G)
        return [G, d, d2]
    got, want = run_both(program)
    np.testing.assert_array_equal(got[0], want[0])
    for g, w in zip(got[1:], want[1:]):
        np.testing.assert_allclose(g, w, rtol=0, atol=8 * np.finfo(dtype).eps)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES[:4])
@pytest.mark.parametrize("dtype", [np.int32, np.float64, np.complex64])
def test_other_windows(shape, dtype):
    """Whole numbers (sums of a few hundred are exact in every type)."""
    def program():
        h = (bh.random.RandomState(4).random123((shape[0] * shape[1],)) % np.uint64(97)).astype(dtype).reshape(shape)
        k = (bh.random.RandomState(5).random123((shape[0] * shape[1],)) % np.uint64(89)).astype(dtype).reshape(shape)
        bh.flush()
        nine = h[1:-1, 1:-1] * 4
        for dr in (0, 1, 2):
            for dc in (0, 1, 2):
                if (dr, dc) != (1, 1):
                    nine = nine + h[dr:shape[0] - 2 + dr, dc:shape[1] - 2 + dc]
        wide = h[3:, 5:] + h[:-3, :-5] + k[3:, :-5] + k[3:, 5:] - h[1:-2, 2:-3] * k[:-3, 4:-1]
        return [nine, wide, h[:, 1:] - h[:, :-1], h[1:] - h[:-1] + k[1:]]
    got, want = run_both(program)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)


@pytest.mark.gpu
def test_repeated_sweeps_equal_single_ones():
    a, b = _grid((1032, 1031), np.float32), _grid((1032, 1031), np.float32)
    workloads.jacobi_repeat(a, 23)
    for _ in range(23):
        d = workloads.jacobi_step(b)
        bh.flush()
        del d
    np.testing.assert_array_equal(a.asnumpy(), b.asnumpy())


DRIVER = r"""
import sys
sys.path.insert(0, %r)
import bohrium_amd as bh
from bohrium_amd import workloads
for n in (512, 2048):
    G = bh.zeros((n, n)); bh.flush(); d = workloads.jacobi_step(G); bh.flush()
"""


def test_small_grids_keep_the_element_walk():
    env = dict(os.environ, BH_HIP_DRY_RUN="1", BH_HIP_DEBUG="2")
    r = subprocess.run([sys.executable, "-c", DRIVER % ROOT], env=env, text=True, stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, timeout=600)
    assert r.returncode == 0, r.stdout[-3000:]
    plans = [("st_h" in p) for p in r.stdout.split("[hip] plan ") if p.startswith("reduce")]
    assert plans == [False, True], plans
