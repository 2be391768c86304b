"""Many one-axis reductions in one flush run as one batched launch of the row skeleton where that is faster than a
segmented launch (or two) each: which flushes do (compile-only), and the sums of both forms (device, against the
oracle)."""
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
def plan(count, rows, cols, f, few=()):
    xs = [bh.empty((rows + 2 * k, cols), np.float32) for k in range(count)] + [bh.empty(s, np.float32) for s in few]
    bh.flush(); bh.message("plan log")
    keep = [f(x) for x in xs]; bh.flush()
    log = [l.split() for l in bh.message("plan log").splitlines() if l.strip()]
    print(sorted(set((l[0], sum(m[0] == l[0] for m in log)) for l in log)), len(set(l[3] for l in log if l[0] == "row")))
for axis in (0, 1):
    plan(60, 300, 320, lambda x: (x * x).sum(axis=axis))                     # one code, one batched launch
    plan(8, 4200, 320, lambda x: (x * x).sum(axis=axis))                     # as many as a batch needs
    plan(7, 4200, 320, lambda x: (x * x).sum(axis=axis))                     # one fewer
    plan(8, 4200, 320, lambda x: (x * x).sum(axis=axis), [(70000, 64), (64, 70000)])   # long ones among them
    plan(8, 2900, 2900, lambda x: (x * x).sum(axis=axis))                    # large enough by themselves
    plan(10, 300, 320, lambda x: x - (x.mean(0)[None, :] if axis == 0 else x.mean(1)[:, None]))
"""


def test_which_flushes_are_batched():
    r = subprocess.run([sys.executable, "-c", DRIVER % ROOT], env=dict(os.environ, BH_HIP_DRY_RUN="1"), text=True,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=600)
    assert r.returncode == 0, r.stdout[-3000:]
    # (skeletons and launches planned, distinct codes of the row skeleton)
    lines = [eval(l.replace("] ", "], ")) for l in r.stdout.splitlines() if l.startswith("[")]
    # (a row's mean is divided in its own loop, a column's in a map)
    for axis, mixed, maps in ((0, [("row", 8), ("seg", 2)], 20), (1, [("row", 9), ("seg", 1)], 10)):
        assert lines[6 * axis:6 * axis + 6] == [
            ([("row", 60)], 1), ([("row", 8)], 1), ([("seg", 7)], 0), (mixed, 1), ([("seg", 8)], 0),
            ([("map", maps), ("row", 10)], 1)], lines


@pytest.mark.gpu
@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("count", [7, 20])
def test_results(axis, count):
    def programs():
        xs = [((bh.arange((300 + 3 * k) * 321) * 7919) % 1009).astype(np.float64).reshape((300 + 3 * k, 321)) for k in range(count)]
        xs += [((bh.arange(70001 * 5) * 31) % 1009).astype(np.float64).reshape((70001, 5) if axis == 0 else (5, 70001))]
        bh.flush()
        return [(x + 1).sum(axis=axis) for x in xs] + [x.max(axis=axis) for x in xs] + [x.sum(axis=axis) * 2 + x.min(axis=axis) for x in xs]
    got, want = run_both(programs)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)  # (whole numbers below 2^53 in any order)
