"""The library's compiled kernels: none spills registers, and every DPP operand has the two wait states that it needs
after a VALU write (the hardware does not wait; the compiler counts them for its own instructions, but not for
the assembler forms of the tile factor, whose operands it could also move)."""
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


def _registers(operand):
    m = re.match(r"-?\|?v(?:(\d+)|\[(\d+):(\d+)\])", operand)
    if not m:
        return []
    return [int(m.group(1))] if m.group(1) else list(range(int(m.group(2)), int(m.group(3)) + 1))


def dpp_hazards(lines):
    """(number of DPP instructions, those that read a register less than two wait states after a VALU write)."""
    written = {}  # register -> wait states since a VALU instruction wrote it
    count, bad = 0, []
    for line in lines:
        m = re.match(r"\s*([vs]_\w+|ds_\w+|buffer_\w+|global_\w+|flat_\w+|scratch_\w+)\s*(.*?)\s*(?://.*)?$", line)
        if not m:
            continue
        op, operands = m.group(1), [x.strip() for x in m.group(2).split(",")]
        if "_dpp" in op:
            count += 1
            source = operands[1].split()[0] if len(operands) > 1 else ""
            if any(written.get(r, 9) < 2 for r in _registers(source)):
                bad.append(line.strip())
        passed = int(operands[0], 0) + 1 if op == "s_nop" else 1
        written = {r: n + passed for r, n in written.items() if n + passed < 2}
        if op.startswith("v_") and not op.startswith("v_mfma"):
            for r in _registers(operands[0]) + (_registers(operands[1]) if "swap" in op else []):
                written[r] = 0
    return count, bad


def test_dpp_hazards_are_seen():
    broadcast = "v_fmac_f64_dpp v[2:3], v[4:5], v[6:7] row_newbcast:3 row_mask:0xf bank_mask:0xf"
    copy = "v_mov_b32_e32 v5, v9"
    for before, hazard in (([copy], True), ([copy, "s_nop 0"], True), ([copy, "s_nop 1"], False),
                           ([copy, "v_add_u32_e32 v1, v1, v1"], True), ([copy, "v_add_u32_e32 v1, v1, v1"] * 1 + ["s_nop 0"], False),
                           (["v_permlane16_swap_b32_e32 v11, v4", "v_add_u32_e32 v1, v1, v1"], True),
                           (["v_mov_b32_e32 v6, v9"], False), (["v_mov_b32_e32 v2, v9"], False)):
        assert dpp_hazards(["s_nop 7"] + before + [broadcast]) == (1, [broadcast] if hazard else [])


def test_dpp_operands_have_their_wait_states(code_objects):
    broadcasts = 0
    for path in code_objects:
        text = subprocess.run([f"{LLVM}/llvm-objdump", "-d", "--no-show-raw-insn", path], check=True, capture_output=True,
                              text=True).stdout
        broadcasts += text.count("row_newbcast")
        assert dpp_hazards(text.splitlines())[1] == []
    assert broadcasts > 1000  # the tile factor's
