"""Large results are stored past the caches: which stores are (compile-only, in the generated source), and that the
values are all there, for every element size, flat, transposed, in place and scanned, and the next kernel and
the host read them."""
import os
import subprocess
import sys

import numpy as np
import pytest

import bohrium_amd as bh

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
M = 1 << 20

# name: (program over the large arrays, whether it stores past the caches)
PROGRAMS = {
    "flat": ("f * 2 + 1", True),
    "a small result": ("f[:31 * M] * 2", False),
    "large enough": ("f[:32 * M] * 2", True),
    "below the limit": ("b[:47 * M].astype(np.float32)", False),
    "above the limit": ("b[:49 * M].astype(np.float32)", True),
    "in place, 192 MiB": ("f[:48 * M].__imul__(2)", False),
    "double, 16 bytes a lane": ("unrolled(2, lambda: d * 2)", True),
    "double, 32 bytes a lane": ("unrolled(4, lambda: d * 2)", False),
    "strided": ("put(f[::8], f[:8 * M] * 2)", False),
    "strided, large": ("put(h[::2], f * 2)", False),
    "transposed": ("put(g.T, q * 2)", False),
    "a column": ("put(g[:, 0], q[:, 0] * 2)", False),
    "narrow rows": ("put(h.reshape((2 * M, 64))[:, :32], f.reshape((2 * M, 32)) * 2)", False),
    "wide rows": ("put(h.reshape((2048, 65536))[:, :32768], f.reshape((2048, 32768)) * 2)", True),
    "offset": ("put(h[1:64 * M + 1], f * 2)", True),
    "transposed operand": ("g.T + q", True),
    "generated": ("bh.arange(128 * M).astype(np.float32)", False),
    "from bytes": ("b.astype(np.float32) + 1", True),
    "complex": ("c + c", False),
    "scan": ("(f > 0).astype(np.int64).cumsum()", True),
    "strided scan": ("put(k[::2], f.cumsum())", False),
    "column sums and their map": ("g - g.sum(axis=0)[None, :]", True),
}

DRIVER = r"""
import sys
sys.path.insert(0, %r)
import numpy as np, bohrium_amd as bh
M = 1 << 20
f, h, d = bh.empty((64 * M,), np.float32), bh.empty((128 * M,), np.float32), bh.empty((64 * M,), np.float64)
g, q = bh.empty((8192, 8192), np.float32), bh.empty((8192, 8192), np.float32)
b, c, k = bh.empty((128 * M,), np.int8), bh.empty((32 * M,), np.complex64), bh.empty((128 * M,), np.float32)
bh.flush()
def put(view, value):
    view[...] = value
    return view
def unrolled(u, fn):
    bh.message("codegen: map_unroll=%%d" %% u)
    y = fn()
    bh.flush()
    bh.message("codegen: map_unroll=4")
    return y
for name, program in %r:
    print("PROGRAM " + name, file=sys.stderr, flush=True)
    keep = eval(program)
    bh.flush()
    del keep
"""


def test_which_stores_go_past_the_caches():
    # (without twins: their first exchange copies the whole array)
    progs = [(n, p) for n, (p, _) in PROGRAMS.items()]
    r = subprocess.run([sys.executable, "-c", DRIVER % (ROOT, progs)], env=dict(os.environ, BH_HIP_DRY_RUN="1", BH_HIP_DEBUG="2", BH_HIP_TWIN_UPDATES="false"),
                       text=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=600)
    assert r.returncode == 0, r.stdout[-3000:]
    got = {}
    for part in r.stdout.split("PROGRAM ")[1:]:
        got[part.splitlines()[0]] = "__builtin_nontemporal_store" in part
    assert got == {n: s for n, (_, s) in PROGRAMS.items()}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.bool_, np.int8, np.int16, np.float32, np.float64, np.complex64])
def test_maps(dtype):
    n = (168 << 20) // np.dtype(dtype).itemsize + 5
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


@pytest.mark.gpu
def test_transposed_scanned_and_in_place():
    r, c = 6501, 6803
    h = (np.arange(r * c) % 1009).astype(np.float32).reshape(r, c)
    x = bh.array(h)
    np.testing.assert_array_equal((x.T + 1).asnumpy(), h.T + 1)
    n = (240 << 20) // 8 + 3
    b = bh.array((np.arange(n) % 3 == 0).astype(np.float32))
    np.testing.assert_array_equal((b > 0).astype(np.int64).cumsum().asnumpy(), np.cumsum(np.arange(n) % 3 == 0))
    x[1:-1, 1:-1] = (x[:-2, 1:-1] + x[2:, 1:-1] + x[1:-1, 2:]) * 0.5
    bh.flush()
    want = h.copy()
    want[1:-1, 1:-1] = (h[:-2, 1:-1] + h[2:, 1:-1] + h[1:-1, 2:]) * np.float32(0.5)
    np.testing.assert_array_equal(x.asnumpy(), want)
