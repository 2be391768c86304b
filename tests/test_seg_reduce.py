"""Segmented reductions (one axis of a large array) against the oracle: the skeleton's edges are the vector
width (contiguous axes of 4k, 2k and odd length), the split of the reduced axis (one piece, several, a
short last piece), lane groups of 4 to 256 and their tails, and what follows the sums."""
import os
import subprocess
import sys

import numpy as np
import pytest

import bohrium_amd as bh
from tests.helpers import run_both

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# (rows, cols): outputs 1 element past a thread's or workgroup's share, reduced lengths 1 past a piece
COLUMNS = [(70001, 1 + 8), (4099, 46), (2050, 500), (129, 4096), (16, 8193), (33, 65537),
           (2050, 513), (1027, 2049)]
ROWS = [(9, 70001), (46, 4099), (500, 2050), (4096, 129), (8193, 16), (65537, 33), (3, 262144 + 3)]


def _input(shape, dtype, seed=5):
    """An array in memory (flushed: the reductions read it, they do not compute it)."""
    n = int(np.prod(shape))
    r = bh.random.RandomState(seed).random123((n,))
    dtype = np.dtype(dtype)
    if dtype == np.bool_:
        x = ((r % np.uint64(97)) != 0).reshape(shape)
    elif dtype.kind in "iu":
        x = (r % np.uint64(100)).astype(dtype).reshape(shape)
    else:
        x = (r % np.uint64(1 << 20)).astype(np.float64) * (2.0 ** -19) - 1.0
        x = (x * 1j + x * 0.5 if dtype.kind == "c" else x).astype(dtype).reshape(shape)
    bh.flush()
    return x


def _bound(got, want, terms, eps, scale):
    """Two sums of `terms` terms of size at most `scale` in any order: each within (terms - 1) eps scale terms / 2 of
    the exact one in the worst case; rounding errors are signed, so sqrt(terms) with a factor of 8 holds them."""
    np.testing.assert_allclose(got, want, rtol=0, atol=8 * eps * scale * terms ** 0.5 * np.log2(terms + 1))


@pytest.mark.gpu
@pytest.mark.parametrize("axis,shape", [(0, s) for s in COLUMNS] + [(1, s) for s in ROWS])
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int64])
def test_sum_and_extremes(axis, shape, dtype):
    n = shape[axis]

    def program():
        x = _input(shape, dtype)
        return [x.sum(axis=axis), (x * x + 1).max(axis=axis), x.min(axis=axis)]
    got, want = run_both(program)
    if np.dtype(dtype).kind == "i":
        np.testing.assert_array_equal(got[0], want[0])
    else:
        _bound(got[0], want[0], n, np.finfo(dtype).eps, 1.0)
    for g, w in zip(got[1:], want[1:]):
        np.testing.assert_allclose(g, w, rtol=np.finfo(dtype).eps * 2 if np.dtype(dtype).kind == "f" else 0)


@pytest.mark.gpu
@pytest.mark.parametrize("axis,shape", [(0, (20011, 12)), (1, (12, 20011)), (1, (5003, 40)), (0, (1024, 514)), (0, (2049, 514))])
@pytest.mark.parametrize("dtype", [np.bool_, np.uint8, np.int16, np.complex64, np.complex128])
def test_other_types(axis, shape, dtype):
    def program():
        x = _input(shape, dtype)
        if np.dtype(dtype) == np.bool_:
            return [x.any(axis=axis), x.all(axis=axis), x.sum(axis=axis)]
        return [x.sum(axis=axis), (x + x).sum(axis=axis)]
    got, want = run_both(program)
    for g, w in zip(got, want):
        if np.dtype(dtype).kind == "c":
            eps = np.finfo(dtype).eps
            _bound(g.real, w.real, shape[axis], eps, 2.0)
            _bound(g.imag, w.imag, shape[axis], eps, 2.0)
        else:
            np.testing.assert_array_equal(g, w)


@pytest.mark.gpu
def test_few_rows_in_one_piece():
    """17 rows of 2^21 + 4 float32: segmented without a split; whole numbers, so the sums are exact."""
    def program():
        x = _input((17, (1 << 21) + 4), np.int32).astype(np.float32)
        bh.flush()
        return [x.sum(axis=0), x.min(axis=0)]
    got, want = run_both(program)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)


@pytest.mark.gpu
@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("shape", [(3001, 64), (64, 3001), (300, 301), (4101, 66), (2050, 513), (33, 65537)])
def test_written_and_following_work(axis, shape):
    """The loop also writes an array, the output is used after the sum, and the input is a strided, reversed or
    transposed view."""
    def program():
        big = _input((2 * shape[0], 2 * shape[1]), np.float64)
        x = big[::2, ::-2]
        m = x.mean(axis)
        c = x - (m[None, :] if axis == 0 else m[:, None])
        v = (c * c).mean(axis)
        s = bh.sqrt(v + 1e-3)
        y = _input(shape[::-1], np.float64, 9).T
        return [m, c, v, s, y.sum(axis=axis) * 2.0 + m, (y * x).max(axis=axis)]
    got, want = run_both(program)
    for g, w in zip(got, want):
        _bound(g, w, shape[axis], np.finfo(np.float64).eps, 4.0)


# More axes: shape, axis, the skeletons of the sum.  (The first axis of three or more is summed by one thread: the fuser
# leaves its loop outside, and that form is no segmented reduction.)
MORE_AXES = [((7, 300, 40), 1, ["row"]), ((7, 4100, 40), 1, ["seg"]), ((7, 4100, 41), 1, ["seg"]), ((7, 40, 300), 2, ["seg"]),
             ((40, 9, 300), 0, ["map", "serial"]), ((5, 3, 70, 70), 2, ["row"]), ((5, 3, 4100, 12), 2, ["seg"]),
             ((5, 3, 12, 4100), 3, ["seg"])]


def test_which_skeletons_more_axes_have():
    prog = DRIVER.split("x = bh.empty")[0] % ROOT + """
for shape, axis in %r:
    x = bh.empty(shape, np.float32); bh.flush()
    print(plan(lambda: x.sum(axis=axis)))
""" % [m[:2] for m in MORE_AXES]
    r = subprocess.run([sys.executable, "-c", prog], env=dict(os.environ, BH_HIP_DRY_RUN="1"), text=True,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=600)
    assert r.returncode == 0, r.stdout[-3000:]
    assert [eval(l) for l in r.stdout.splitlines() if l.startswith("[")] == [m[2] for m in MORE_AXES], r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("shape,axis", [m[:2] for m in MORE_AXES])
def test_more_axes(shape, axis):
    def program():
        x = _input(shape, np.float32)
        return [x.sum(axis=axis), x.max(axis=axis)]
    got, want = run_both(program)
    _bound(got[0], want[0], shape[axis], np.finfo(np.float32).eps, 1.0)
    np.testing.assert_array_equal(got[1], want[1])


@pytest.mark.gpu
def test_infinities_nans_and_repeats():
    """Infinities and NaNs stay in their own output; a repeated body gives the same sums from a replayed graph."""
    h = np.ones((4096, 40), np.float32)
    h[5, 3], h[6, 7], h[7, 9] = np.inf, -np.inf, np.nan
    x = bh.array(h)
    s = x.sum(axis=0).asnumpy()
    assert s[3] == np.inf and s[7] == -np.inf and np.isnan(s[9])
    np.testing.assert_array_equal(np.delete(s, [3, 7, 9]), np.full(37, 4096.0, np.float32))
    t = bh.ones((8192, 33), np.float64)
    acc = bh.zeros((33,), np.float64)

    def body():
        acc[...] = acc + t.sum(axis=0)
    bh.do_while(body, 20)
    np.testing.assert_array_equal(acc.asnumpy(), np.full(33, 20 * 8192.0))


DRIVER = r"""
import sys
sys.path.insert(0, %r)
import numpy as np, bohrium_amd as bh
def plan(f):
    bh.flush(); bh.message("plan log"); keep = f(); bh.flush()
    return [l.split()[0] for l in bh.message("plan log").splitlines() if l.strip()]
x = bh.empty((4096, 512), np.float32)
print(plan(lambda: x.sum(axis=0)), plan(lambda: x.sum(axis=1)), plan(lambda: x.T.sum(axis=0)))
print(plan(lambda: x[:64, :64].sum(axis=0)), plan(lambda: x[:64, :64].sum(axis=1)))
for dtype, shape in (("float32", (2048, 256)), ("float32", (512, 2048)), ("float32", (1023, 2049)), ("float32", (2048, 512)),
                     ("float32", (4096, 16)), ("float32", (4095, 16)), ("float32", (32, 65536)), ("float32", (32, 65535)),
                     ("float32", (31, 1 << 18)), ("float32", (31, 1 << 21)), ("float64", (31, 1 << 21)), ("float32", (16, 4097))):
    y = bh.empty(shape, dtype); bh.flush()
    print(plan(lambda: y.sum(axis=0)) + plan(lambda: y.T.sum(axis=1)))
y, z = bh.empty((4096, 512), np.float32), bh.empty((4096, 512), np.float32); bh.flush()
for r in (1360, 1366, 1400):  # three arrays: 2^21 loads are 1365.3 rows
    print(plan(lambda: (x[:r] * y[:r] + z[:r]).sum(axis=0)) + plan(lambda: (x[:r] * 2 + x[:r]).sum(axis=0)))
print(plan(lambda: x[:256, :256].mean(axis=0)), plan(lambda: x[:128, :128].mean(axis=0)), plan(lambda: x[:31].mean(axis=0)))
bh.message("codegen: row_reduce=0")
print(plan(lambda: x.sum(axis=1)))
"""


def test_which_reductions_are_segmented():
    r = subprocess.run([sys.executable, "-c", DRIVER % ROOT], env=dict(os.environ, BH_HIP_DRY_RUN="1"), text=True,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=600)
    assert r.returncode == 0, r.stdout[-3000:]
    lines = [l for l in r.stdout.splitlines() if l.startswith("[")]
    # (columns: many rows or many elements, below 32 rows only by 16-byte loads in one launch)
    row, seg, plain = "['row', 'row']", "['seg', 'seg']", "['map', 'map']"
    assert lines == ["['seg'] ['seg'] ['seg']", "['row'] ['row']", row, row, row, seg, seg, row, seg, row, plain, seg, plain, plain,
                     row, "['seg', 'row']", "['seg', 'row']", "['seg'] ['row', 'map'] ['map', 'map']", "['map']"], r.stdout
