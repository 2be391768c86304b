"""The persistent launch links every code of a flush into one kernel, so their LDS tiles add up: a flush of several
tiled maps that do not fit together runs as levels, one whose tiles fit as one persistent kernel (compile-only,
and on the device against the oracle)."""
import os
import subprocess
import sys

import numpy as np
import pytest

import bohrium_amd as bh
from tests.helpers import run_both

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
import numpy as np, bohrium_amd as bh
def program(xs, ys, codes):
    # ten maps of one code (a batch group) and `codes` maps of transposes, each a code of its own
    out = [x + 1 for x in xs]
    for k in range(codes):
        t = ys[k].T
        for _ in range(k):
            t = t * 3
        out.append(t + 5)
    return out
"""

DRIVER = r"""
import sys
sys.path.insert(0, %r)
exec(%r)
from bohrium_amd import _bh_api
_bh_api.set_flush_threshold(10 ** 7)
bh.message("batch_persistent: on")
xs = [bh.empty((3000 + k,), np.float64) for k in range(10)]
ys = [bh.empty((1100, 1200 + 16 * k), np.float64) for k in range(7)]
bh.flush()
keep = program(xs, ys, %d); bh.flush()
"""


@pytest.mark.parametrize("codes,fits", [(1, True), (2, True), (3, False), (7, False)])
def test_the_tiles_of_all_codes_have_to_fit(tmp_path, codes, fits):
    """Every code here has one 64 x 65 tile of float64 (33,280 bytes); half of a CU's LDS holds two of them."""
    env = dict(os.environ, BH_HIP_DRY_RUN="1", BH_HIP_DUMP_DIR=str(tmp_path))
    r = subprocess.run([sys.executable, "-c", DRIVER % (ROOT, PROGRAM, codes)], env=env, text=True, stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, timeout=600)
    assert r.returncode == 0, r.stdout[-3000:]
    heads = [f.read_text().splitlines()[0] for f in sorted(tmp_path.glob("persist_*.txt"))]
    assert heads, r.stdout
    assert (heads[-1] != "persistent none") == fits, heads


@pytest.mark.gpu
@pytest.mark.parametrize("codes,launches", [(2, 1), (7, 0)])
def test_results(codes, launches):
    env = {}
    exec(PROGRAM, env)

    def count():
        return int([l for l in bh.message("statistic").splitlines() if l.startswith("persist_launches")][0].split()[1])

    def programs():
        xs = [bh.arange(3000 + k).astype(np.float64) for k in range(10)]
        ys = [bh.arange(1100 * (1200 + 16 * k)).astype(np.float64).reshape((1100, 1200 + 16 * k)) for k in range(7)]
        bh.flush()  # (the inputs are a flush of their own, persistent or not)
        before.append(count())
        return env["program"](xs, ys, codes)
    before = []
    bh.message("batch_persistent: on")
    try:
        got, want = run_both(programs)
        assert count() - before[0] == launches
    finally:
        bh.message("batch_persistent: off")
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)
