"""Registers and memory of the built kernels, from the metadata of the code
objects in libsporder_hip.so: bounds that their speed was measured with and
that a change elsewhere in a shared header can lose without a wrong result."""

import re
import shutil
import subprocess

import pytest

from chunkedgreedy_amd import build

LLVM = "/opt/rocm/llvm/bin"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{mangled name: metadata} of every kernel of the library."""
    if not build.LIB_PATH.exists():
        pytest.fail("libsporder_hip.so is not built")
    where = tmp_path_factory.mktemp("code_objects")
    lib = shutil.copy(build.LIB_PATH, where)
    subprocess.run([f"{LLVM}/llvm-objdump", "--offloading", lib], check=True,
                   capture_output=True, cwd=where)
    found = {}
    for obj in where.glob("*gfx950*"):
        notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", str(obj)], check=True,
                               capture_output=True, text=True).stdout
        # One list entry of amdhsa.kernels per kernel; its keys are sorted.
        for entry in re.split(r"\n  - \.agpr_count:", notes)[1:]:
            numbers = {k: int(v) for k, v in re.findall(r"\n    \.(\w+): +(\d+)", entry)}
            found[re.search(r"\n    \.symbol: +'?([^'\s]+?)\.kd", entry)[1]] = numbers
    return found


@pytest.mark.parametrize("cells", range(5, 17))
def test_uncounted_global_sketch_spills_nothing(kernels, cells):
    name = [k for k in kernels if f"ovf_sketch_kernelILi{cells}ELb0ELb0E" in k]
    assert len(name) == 1
    k = kernels[name[0]]
    assert k["private_segment_fixed_size"] == 0
    assert k["sgpr_spill_count"] == 0 and k["vgpr_spill_count"] == 0
    assert k["vgpr_count"] <= 80 # 6 waves per SIMD
