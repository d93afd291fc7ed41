"""csrc/check_registers.py, which the build runs over the kernels that read LDS and multiply through inline asm: what it lets
pass and what it stops, on listings with a mistake planted in them."""
import os
import subprocess
import sys

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "aitemplate_amd", "csrc")
sys.path.insert(0, CSRC)
import check_registers  # noqa: E402

WIDE, ROWS, OTHER = "_gemm_rcr_wide_kernel_x", "_gemm_rcr_rows_kernel_x", "_gemm_rcr_dma_kernel_x"

# a loop of one step: fragments read, multiplied and, behind the wait, read for the next turn
LOOP = """
ds_read_b128 v[4:7], v0
ds_read_b128 v[8:11], v0 offset:1024
s_waitcnt lgkmcnt(0)
v_mfma_f32_16x16x32_f16 a[0:3], v[4:7], v[8:11], 0
ds_read_b128 v[12:15], v0 offset:2048
v_add_u32 v1, v2, v3
s_waitcnt lgkmcnt(0)
v_mfma_f32_16x16x32_f16 a[0:3], v[12:15], v[8:11], a[0:3]
ds_read_b128 v[4:7], v0 offset:4096
s_cbranch_scc1 @2
s_nop 15
s_nop 3
s_waitcnt lgkmcnt(0)
v_accvgpr_read_b32 v20, a0
scratch_store_dwordx4 off, v[4:7], off
s_endpgm
"""


def _listing(text, symbol=WIDE):
    """As llvm-objdump writes it; @n branches to line n."""
    out = [f"0000000000001000 <{symbol}>:"]
    for i, line in enumerate(text.strip().splitlines()):
        target = ""
        if "@" in line:
            line, to = line.split("@")
            line, target = line + "7", f" <{symbol}+0x{8 * int(to):x}>"
        out.append(f"\t{line:<60}// {0x1000 + 8 * i:012X}: BF800000{target}")
    return "\n".join(out)


def _faults(text, symbol=WIDE):
    (name, body), = check_registers.parse(_listing(text, symbol)).items()
    return check_registers.check(body, bool(check_registers.MULTIPLY.search(name)))


def test_a_sound_loop_passes():
    assert _faults(LOOP) == []


@pytest.mark.parametrize("old,new,named", [
    ("v_add_u32 v1, v2, v3", "v_mov_b32 v20, v13", "v13"),                           # a copy of what has not arrived
    ("v_add_u32 v1, v2, v3", "scratch_store_dwordx4 off, v[14:17], off", "v14"),     # a spill
    ("v_add_u32 v1, v2, v3", "v_mov_b32 v15, v2", "v15"),                            # a write that the read overtakes
    ("s_waitcnt lgkmcnt(0)\nv_mfma_f32_16x16x32_f16 a[0:3], v[12:15]",
     "s_waitcnt lgkmcnt(1)\nv_mfma_f32_16x16x32_f16 a[0:3], v[12:15]", "v12"),       # a wait that is none
    ("s_nop 3\ns_waitcnt lgkmcnt(0)", "s_nop 3", "v4"),                              # none behind the loop
    ("s_nop 15\ns_nop 3", "s_nop 8", "a0"),                                          # results taken early
    ("s_waitcnt lgkmcnt(0)\nv_mfma_f32_16x16x32_f16 a[0:3], v[4:7]", "v_mfma_f32_16x16x32_f16 a[0:3], v[4:7]", "v4"),
])
def test_planted_mistakes_are_found(old, new, named):
    assert old in LOOP
    found = _faults(LOOP.replace(old, new, 1))
    assert any(f" names {named} " in fault for fault in found), found


def test_a_read_is_followed_over_the_back_edge():
    """The turn's last read is named by the next turn's first instruction; in a straight line nothing names it."""
    loop = LOOP.replace("s_waitcnt lgkmcnt(0)\nv_mfma_f32_16x16x32_f16 a[0:3], v[4:7]",
                        "s_waitcnt lgkmcnt(0)\nv_mov_b32 v30, v31\nv_mfma_f32_16x16x32_f16 a[0:3], v[4:7]")
    assert _faults(loop) == []                                          # (the loop starts with its wait)
    found = _faults(loop.replace("@2", "@3"))                           # it starts behind the wait
    assert any(" names v4 " in fault for fault in found), found


def test_waits_count_the_younger_operations():
    """lgkmcnt(1) lets the youngest operation be outstanding: the read before it has arrived."""
    text = "ds_read_b128 v[4:7], v0\nds_read_b128 v[8:11], v0\ns_waitcnt lgkmcnt(1)\nv_mov_b32 v1, {}\ns_endpgm"
    assert _faults(text.format("v4")) == []
    assert _faults(text.format("v8")) != []


def test_which_kernels_are_looked_at():
    early = LOOP.replace("s_nop 15\ns_nop 3", "s_nop 8")
    assert _faults(early, ROWS) == []                                   # (its products are the compiler's own)
    assert _faults(LOOP.replace("v_add_u32 v1, v2, v3", "v_mov_b32 v20, v13"), ROWS) != []
    assert check_registers.parse(_listing(early, OTHER)) == {}


def test_what_cannot_be_followed_is_an_error():
    with pytest.raises(ValueError, match="not followed"):
        check_registers.parse(_listing("s_swappc_b64 s[30:31], s[0:1]\ns_endpgm"))


def test_the_build_runs_it():
    out = subprocess.run(["make", "-B", "-n", "-C", CSRC, f"PYTHON={sys.executable}"], text=True, stdout=subprocess.PIPE, check=True).stdout
    assert out.count("check_registers.py build/gemm_inst_") == 36
