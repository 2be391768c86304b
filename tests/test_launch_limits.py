"""A launch has fewer than 2^32 threads: plans of very large arrays stay below that (compile-only, no array is ever
allocated), and the launch entry refuses what does not, before it reaches the runtime."""
import ctypes
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
import sys
sys.path.insert(0, %r)
import numpy as np, bohrium_amd as bh
for shape, axis, dtype in %r:
    x = bh.empty(shape, np.dtype(dtype))
    bh.flush(); bh.message("plan log")
    keep = x.max(axis=axis); bh.flush()
    print([l.split()[:2] for l in bh.message("plan log").splitlines() if l.strip()])
    del keep, x
"""
# (rows of 16 elements: 64 outputs a workgroup, 2^30 of them are 2^24 workgroups of 256 threads)
SHAPES = [((1 << 30, 16), 1, "int8"), (((1 << 31) - 1, 16), 1, "int8"), (((1 << 30) - 64, 16), 1, "int8"),
          ((16, (1 << 31) - 1), 0, "int8"), ((40, 1 << 30), 0, "float64")]


def test_reductions_of_many_outputs():
    r = subprocess.run([sys.executable, "-c", DRIVER % (ROOT, SHAPES)], env=dict(os.environ, BH_HIP_DRY_RUN="1"), text=True,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=600)
    assert r.returncode == 0, r.stdout[-3000:]
    plans = [eval(l) for l in r.stdout.splitlines() if l.startswith("[")]
    assert len(plans) == len(SHAPES), r.stdout
    for shape, plan in zip(SHAPES, plans):
        for strategy, grid in plan:
            assert int(grid) * 256 < 1 << 32, (shape, strategy, grid)
    # one workgroup below the limit the segmented skeleton still runs, at it the capped walk does
    assert plans[0] == [["map", "2048"]] and plans[2] == [["seg", str((1 << 24) - 1)]], plans


@pytest.mark.parametrize("grid,block", [(1 << 24, 256), (1 << 26, 64), (1 << 31, 1)])
def test_the_launch_entry_refuses_too_many_threads(grid, block):
    hip = ctypes.CDLL(os.path.join(ROOT, "bohrium_amd", "lib", "libbh_ve_hip.so"))
    hip.bhhip_last_error.restype = ctypes.c_char_p
    hip.bhhip_launch.argtypes = [ctypes.c_void_p, ctypes.c_uint64, ctypes.c_uint32, ctypes.c_void_p, ctypes.c_size_t]
    assert hip.bhhip_launch(None, grid, block, None, 0) != 0
    assert b"grid too large" in hip.bhhip_last_error()
