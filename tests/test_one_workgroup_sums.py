"""Full reductions that one workgroup finishes without a finalize launch: lengths around one workgroup's share
(1024 elements) and beyond, with scalar work behind the sum that is kept, repeated or batched, and with a
following block that reads what the loop wrote (which keeps its finalize)."""
import os
import subprocess
import sys

import numpy as np
import pytest

import bohrium_amd as bh
from tests.helpers import run_both

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 3, 255, 256, 257, 1023, 1024, 1025, 4097])
def test_sums_and_tails(n):
    def program():
        x = (bh.random.RandomState(n).random123((n,)) % np.uint64(1000)).astype(np.float64)
        bh.flush()
        out = bh.zeros((4,))
        y = x * 2
        out[1] = y.sum() * 3 + 1
        out[2] = (x.max() + out[1]) * 2
        bh.flush()
        z = x + 1
        s = z.sum()
        w = z[: min(n, 9)] * s      # reads what the loop wrote
        return [out, y, (x > 500).astype(np.int64).sum(), w, x.min()]
    got, want = run_both(program)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)  # (whole numbers below 2^53)


@pytest.mark.gpu
def test_repeated_and_batched():
    acc = bh.zeros((1,))
    x = bh.ones((700,))

    def body():
        acc[...] = acc + x.sum()
    bh.do_while(body, 25)
    assert float(acc.asnumpy()[0]) == 25 * 700
    xs = [bh.ones((n,)) for n in list(range(200, 2200, 100)) + [600, 1024, 1025]]
    bh.flush()
    sums = [(x * 2).sum() + 1 for x in xs]
    for s, x in zip(bh.asnumpy_many(sums), xs):
        assert float(s) == 2 * x.size + 1


DRIVER = r"""
import sys
sys.path.insert(0, %r)
import bohrium_amd as bh
def launches(f):
    a = [l for l in bh.message("statistic").splitlines() if l.startswith("launches:")][0]
    keep = f(); bh.flush()
    b = [l for l in bh.message("statistic").splitlines() if l.startswith("launches:")][0]
    return int(b.split()[1]) - int(a.split()[1])
x, y = bh.empty((1000,)), bh.empty((5000,)); bh.flush()
print(launches(lambda: (x * 2).sum()), launches(lambda: (y * 2).sum()))
"""


def test_planned_launches():
    r = subprocess.run([sys.executable, "-c", DRIVER % ROOT], env=dict(os.environ, BH_HIP_DRY_RUN="1"), text=True,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=600)
    assert r.returncode == 0, r.stdout[-3000:]
    assert r.stdout.split() == ["1", "2"], r.stdout
