"""The tile kernels of the matrix products load the next K step while the current one runs on the matrix cores: in
the disassembly of their main loops every global load stands before the first product (a load behind the products is
waited for right after, and nothing runs beside it)."""
import os
import shutil
import subprocess

import pytest

from tests.test_kernel_barriers import OBJDUMP, ROOT, _instructions

pytestmark = pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="ROCm llvm-objdump not installed")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    d = tmp_path_factory.mktemp("gemm")
    shutil.copy(os.path.join(ROOT, "bohrium_amd", "lib", "libbh_blas_hip.so"), d)
    subprocess.run([OBJDUMP, "--offloading", "libbh_blas_hip.so"], cwd=d, check=True, stdout=subprocess.DEVNULL)
    code = [f for f in os.listdir(d) if f.endswith("gfx950")]
    assert len(code) == 1, code
    text = subprocess.run([OBJDUMP, "-d", code[0]], cwd=d, check=True, stdout=subprocess.PIPE, text=True).stdout
    out = {}
    for sym, at, ins, target in _instructions(text):
        out.setdefault(sym, []).append((at, ins, target))
    return out


def _main_loop(code):
    """The instructions from the target of the first backward branch over products and a barrier to that branch."""
    for at, ins, target in code:
        if target is None or target >= at or not ins.startswith(("s_branch", "s_cbranch")):
            continue
        body = [i for a, i, _ in code if target <= a <= at]
        if any("v_mfma" in i for i in body) and any(i.startswith("s_barrier") for i in body):
            return body
    return None


@pytest.mark.parametrize("kernel,element", [("gemm_mfma", "f"), ("gemm_mfma", "d"), ("gemm_complex", "f"), ("gemm_complex", "d")])
def test_loads_stand_before_the_products(kernels, kernel, element):
    names = [k for k in kernels if kernel + "I" + element in k]
    assert len(names) >= 6, sorted(kernels)
    for name in names:
        body = _main_loop(kernels[name])
        assert body is not None, name
        first = [n for n, i in enumerate(body) if "v_mfma" in i][0]
        loads = [n for n, i in enumerate(body) if i.startswith("global_load")]
        assert loads and max(loads) < first, (name, loads, first)
