"""Registers of the gradient kernel's variants, as the built library's own code object states them:
a variant for more waves per SIMD is of use only while its registers are not spilled to memory (in fp32;
fp64's accumulators alone exceed what seven or eight waves leave)."""

from __future__ import annotations

import os
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from autan_amd import build

LLVM = Path(os.environ.get("ROCM_PATH", "/opt/rocm")) / "llvm" / "bin"


def spills(lib: Path, tmp: Path) -> dict[str, int]:
    """Spilled vector registers by mangled kernel name."""
    fat, code = tmp / "fat", tmp / "code"
    subprocess.run(["objcopy", "--dump-section", f".hip_fatbin={fat}", lib, "/dev/null"], check=True)
    subprocess.run([LLVM / "clang-offload-bundler", "--unbundle", "--type=o", f"--input={fat}", f"--output={code}",
                    f"--targets=hipv4-amdgcn-amd-amdhsa--{build.ARCH}"], check=True)
    notes = subprocess.run([LLVM / "llvm-readelf", "--notes", code], check=True, capture_output=True, text=True).stdout
    found = re.findall(r"\.symbol:\s+(\w+)\.kd.*?\.vgpr_spill_count:\s+(\d+)", notes, re.S)
    return {name: int(n) for name, n in found}


@pytest.mark.skipif(shutil.which("objcopy") is None or not (LLVM / "llvm-readelf").exists(), reason="no LLVM tools")
def test_gradient_variants_do_not_spill(tmp_path):
    of = spills(build.PKG / "libmxeuler.so", tmp_path)
    grad = {n: v for n, v in of.items() if "k_grad_lds" in n}
    assert grad
    for name, n in grad.items():
        occupancy = int(re.search(r"Li(\d+)E", name).group(1))
        if occupancy == 0 or (occupancy == 7 and "k_grad_ldsIf" in name):
            assert n == 0, name
        elif "k_grad_ldsIf" in name:
            assert n < 10, name  # 64 registers: a few of the weights' and positions'
