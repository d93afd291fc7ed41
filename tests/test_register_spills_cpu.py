"""Registers that the compiled kernels spill: an argument held in registers over a kernel's main loop, for a use behind it, is
paid for with lane writes and scratch memory around the loop.  The limits are what the kernels had before their coordinates
came from reciprocals, which are arguments too (320 rows: in scratch memory and vector registers)."""
import os
import re
import subprocess

import pytest

from aitemplate_amd import _kernels

LLVM = os.environ.get("ROCM_LLVM_BIN", "/opt/rocm/llvm/bin")
TYPES = r"(?:DF16_|DF16b)"
ATTENTION = r"_ZN6aitamd21attention_pipe_kernelI" + TYPES + r"NS_8AttnPipeI{0}EEEEvNS_10AttnParamsE"
PERSISTENT = r"_ZN6aitamd23gemm_rcr_persist_kernelI" + TYPES + r"NS_15GemmTilePersistI{0}EEENS_8EpilogueILi{1}EEE{2}EEvNS_10GemmParamsE"
ROWS_320 = "Li320ELi256ELi32ELi2ELi4ELi4ELi16ELi320ELi0"

# kernels (regular expression), and the most scratch bytes, scalar and vector registers that one of them may spill
LIMITS = [
    # head dims to 64 (48): four workgroups per CU, waves in two groups, 256 rows, 64 rows
    pytest.param(ATTENTION.format("Li4ELi2ELi1ELi4ELi1ELi1ELi1ELi4E"), 24, 4, 5, id="attention-d64-small"),
    pytest.param(ATTENTION.format("Li3ELi2ELi1ELi4ELi1ELi1ELi1ELi4E"), 8, 0, 1, id="attention-d48-small"),
    pytest.param(ATTENTION.format("Li4ELi2ELi2ELi4ELi1ELi2ELi1ELi2E"), 0, 4, 0, id="attention-d64-groups"),
    pytest.param(ATTENTION.format("Li4ELi2ELi1ELi4ELi2ELi1ELi1ELi2E"), 0, 11, 0, id="attention-d64-rows256"),
    pytest.param(ATTENTION.format("Li4ELi2ELi1ELi2ELi1ELi1ELi1ELi2E"), 0, 12, 0, id="attention-d64-rows64"),
    # 320 x 256, permuted store: K of fewer slabs than the ring has, and more
    pytest.param(PERSISTENT.format(ROWS_320, "[01]", "Lb1ELb1E"), 152, 44, 45, id="gemm-320-rows-permuted-short-k"),
    pytest.param(PERSISTENT.format(ROWS_320, "[01]", "Lb1ELb0E"), 232, 41, 57, id="gemm-320-rows-permuted"),
]


@pytest.fixture(scope="module")
def spills(tmp_path_factory):
    """{kernel: (scratch bytes, scalar, vector registers spilled)} of the built library"""
    if not os.path.exists(f"{LLVM}/llvm-objdump") or not os.path.exists(f"{LLVM}/llvm-readelf"):
        pytest.skip("no llvm-objdump or llvm-readelf")
    tmp = tmp_path_factory.mktemp("code")
    (tmp / "lib.so").symlink_to(_kernels.KERNEL_LIB_PATH)
    subprocess.run([f"{LLVM}/llvm-objdump", "--offloading", str(tmp / "lib.so")], check=True, cwd=tmp, stdout=subprocess.DEVNULL)
    found = {}
    for code in tmp.glob("*gfx950"):
        notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", str(code)], check=True, text=True, stdout=subprocess.PIPE).stdout
        for part in re.split(r"^  - \.", notes, flags=re.M)[1:]:
            value = dict(re.findall(r"\.?(name|private_segment_fixed_size|sgpr_spill_count|vgpr_spill_count): +(\S+)$", part, flags=re.M))
            if len(value) == 4:
                found[value["name"]] = tuple(int(value[k]) for k in ("private_segment_fixed_size", "sgpr_spill_count", "vgpr_spill_count"))
    return found


@pytest.mark.parametrize("kernel,scratch,scalar,vector", LIMITS)
def test_spilled_registers(spills, kernel, scratch, scalar, vector):
    of = {name: s for name, s in spills.items() if re.fullmatch(kernel, name)}
    assert of, "no such kernel in the library"
    over = {name: s for name, s in of.items() if s[0] > scratch or s[1] > scalar or s[2] > vector}
    assert not over
