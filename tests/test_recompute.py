"""Cheap temporaries repeated in front of a later reader (recompute_temporaries): which programs are rewritten
(compile-only: the stored temporary disappears from the planned launches) and that the results do not change
(device: with the rewrite and without it, bit for bit, and against the oracle)."""
import os
import subprocess
import sys

import numpy as np
import pytest

import bohrium_amd as bh
from tests.helpers import run_both

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAMS = r"""
import numpy as np, bohrium_amd as bh
def both(x, axis, keep=False, write=False, square=False):
    m = x.mean(axis)
    e = m[None, :] if axis == 0 else m[:, None]
    c = x * e if square else x - e
    v = (c * c).mean(axis)
    if write:
        m += 1.0
    z = c / (v[None, :] if axis == 0 else v[:, None])
    return [z, v, c] if keep else [z, v]
def centred(x):
    c = x - x.mean()          # the mean is freed before the second reader
    return [c * (c * c).sum(), c.max()]
def from_temp(x):
    t = x * 2.0               # the large input is made in the flush: stored once or not at all
    c = t - t.mean(1)[:, None]
    return [c / c.max(1)[:, None]]
def absolute(x):
    c = bh.abs(x)
    return [c / c.sum(0)[None, :], x.sum()]
"""

DRIVER = r"""
import sys
sys.path.insert(0, %r)
exec(%r)
x = bh.empty((2048, 512), np.float32); bh.flush()
def arrays(f):
    bh.message("plan log")
    keep = f(); bh.flush()
    b = [l for l in bh.message("statistic").splitlines() if l.startswith("recomputed")]
    return int(b[0].split()[1])
print(arrays(lambda: both(x, 1)), arrays(lambda: both(x, 0)), arrays(lambda: both(x, 1, keep=True)),
      arrays(lambda: both(x, 1, write=True)), arrays(lambda: both(x, 1, square=True)), arrays(lambda: centred(x)),
      arrays(lambda: from_temp(x)), arrays(lambda: absolute(x)), arrays(lambda: both(x[:64], 1)))
"""


def test_what_is_rewritten():
    r = subprocess.run([sys.executable, "-c", DRIVER % (ROOT, PROGRAMS)], env=dict(os.environ, BH_HIP_DRY_RUN="1"), text=True,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=600)
    assert r.returncode == 0, r.stdout[-3000:]
    # (the counter runs on: kept, written and multiplied ones, inputs made in the flush and small arrays add nothing)
    assert r.stdout.split() == ["1", "2", "2", "2", "2", "3", "3", "4", "4"], r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_results_do_not_change(dtype):
    env = {}
    exec(PROGRAMS, env)
    h = np.random.RandomState(1).uniform(-3, 5, (2049, 515)).astype(dtype)

    def programs():
        x = bh.array(h)
        bh.flush()
        return (env["both"](x, 1) + env["both"](x, 0) + env["both"](x, 1, keep=True) + env["both"](x, 0, write=True) +
                env["centred"](x) + env["from_temp"](x) + env["absolute"](x))
    bh.message("recompute_temporaries: off")
    plain = [a.asnumpy() for a in programs()]
    bh.message("recompute_temporaries: on")
    got, want = run_both(programs)
    for g, p, w in zip(got, plain, want):
        eps = np.finfo(dtype).eps
        np.testing.assert_array_equal(g, p)
        # sums of up to 2^20 terms of size at most 64, order free: sqrt(terms) eps with a factor of 8
        np.testing.assert_allclose(g, w, rtol=8 * 1024 * eps, atol=8 * 1024 * eps * np.abs(w).max())


def test_a_long_list_is_left_alone():
    """A flush far beyond the flush threshold (thousands of small arrays) is not searched: 1200 arrays of their own sizes
    in front of a program that is rewritten by itself, and 300, which still are a list that is."""
    prog = r"""
import sys
sys.path.insert(0, %r)
exec(%r)
from bohrium_amd import _bh_api
_bh_api.set_flush_threshold(10 ** 7)
x = bh.empty((2048, 512), np.float32)
ys = [bh.empty((256 + k,), np.float32) for k in range(1200)]
bh.flush()
for count in (1200, 300):
    keep = [((y * 2.0 + 1.0).sum()) for y in ys[:count]] + both(x, 1)
    bh.flush()
    print([l for l in bh.message("statistic").splitlines() if l.startswith("recomputed")][0].split()[1])
""" % (ROOT, PROGRAMS)
    r = subprocess.run([sys.executable, "-c", prog], env=dict(os.environ, BH_HIP_DRY_RUN="1"), text=True,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=600)
    assert r.returncode == 0, r.stdout[-3000:]
    assert r.stdout.split() == ["0", "1"], r.stdout


def test_a_freed_input_named_twice_is_freed_once(tmp_path):
    """c = v[:, None] + v[None, :] is repeated behind the free of v: the free moves behind the reader, once."""
    lib, csrc = os.path.join(ROOT, "bohrium_amd", "lib"), os.path.join(ROOT, "bohrium_amd", "csrc")
    exe = str(tmp_path / "recompute_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I" + os.path.join(csrc, "include"), "-I" + csrc,
                    os.path.join(ROOT, "tests", "csrc", "recompute_check.cpp"), os.path.join(csrc, "ve_hip", "rewrite.cpp"),
                    "-o", exe, "-L" + lib, "-lbh", "-Wl,-rpath," + lib], check=True)
    out = subprocess.run([exe], stdout=subprocess.PIPE, text=True, check=True, timeout=60).stdout.splitlines()
    assert out[0] == "rewritten 1", out
    assert out.count("BH_FREE v") == 1, out
    at = [k for k, l in enumerate(out) if l.startswith("BH_DIVIDE z again")]
    assert len(at) == 1 and out[at[0] - 1] == "BH_ADD again v v" and out.index("BH_FREE v") > at[0], out
    assert len(out) == len(set(out)), out
