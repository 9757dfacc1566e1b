"""The library's compiled kernels: none spills registers."""
import glob
import os
import re
import shutil
import subprocess

import pytest

from slamplay_amd import _capi as C

LLVM = "/opt/rocm/llvm/bin"


@pytest.fixture(scope="module")
def code_objects(tmp_path_factory):
    lib = os.path.join(os.path.dirname(C.__file__), "libslamplay_ba.so")
    if not os.path.exists(lib) or not os.path.exists(f"{LLVM}/llvm-objdump"):
        pytest.skip("needs the built library and llvm-objdump")
    out = tmp_path_factory.mktemp("code")
    shutil.copy(lib, out / "lib.so")
    subprocess.run([f"{LLVM}/llvm-objdump", "--offloading", str(out / "lib.so")], check=True, capture_output=True)
    found = sorted(glob.glob(str(out / "*gfx950")))
    assert found
    return found


def _kernels(path):
    """(name, fields) of each kernel in a code object's metadata."""
    text = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", path], check=True, capture_output=True, text=True).stdout
    for block in re.split(r"\n  - (?=\.)", text.split("amdhsa.kernels:")[1])[1:]:
        fields = dict(re.findall(r"^ *(\.\w+): +(\S+)$", block, re.M))
        if ".vgpr_spill_count" in fields:
            yield re.search(r"^ {4}\.name: +(\S+)$", block, re.M).group(1), fields


def test_no_kernel_spills(code_objects):
    kernels = [k for path in code_objects for k in _kernels(path)]
    assert len(kernels) > 100
    spilled = {n: f[".vgpr_spill_count"] for n, f in kernels
               if int(f[".vgpr_spill_count"]) or int(f[".private_segment_fixed_size"])}
    assert spilled == {}
