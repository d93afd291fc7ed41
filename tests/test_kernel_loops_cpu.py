"""The K loops of the 64 x 64 GEMM tiles for operands to transpose, as they were compiled: one straight line with a slab's loads
ahead of its matrix instructions (kLoadsFirst, csrc/gemm_kernel_dma.hpp).  With branches around the loads' offsets, and the loads
behind the instructions, 24 x 64 x 64 x 2048 took 1.14 times as long."""
import os
import re
import subprocess

import pytest

from aitemplate_amd import _kernels

LLVM = os.environ.get("ROCM_LLVM_BIN", "/opt/rocm/llvm/bin")
KERNEL = re.compile(r"^_ZN6aitamd19gemm_rcr_dma_kernelI(DF16_|DF16b)NS_11GemmTileDmaILi64ELi64ELi(64|128)ELi2ELi2ELi4E.*"
                    r"Epilogue.*ELb0ELi([123])EEEvNS_10GemmParamsE$")


def _k_loop(lines):
    """The shortest run of instructions from a branch's target to the branch that multiplies and loads to LDS."""
    at, body, found = {}, [], None
    for line in lines:
        m = re.match(r"^\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+):(.*)$", line)
        if not m:
            continue
        at[int(m[3], 16)] = len(body)
        body.append(f"{m[1]} {m[2]}")
        t = re.search(r"<.*?(?:\+0x([0-9a-f]+))?>", m[4]) if m[1].startswith(("s_branch", "s_cbranch")) else None
        first = at.get(min(at) + int(t[1] or "0", 16)) if t else None
        if first is None:
            continue
        loop = body[first:]
        if (any(i.startswith("v_mfma") for i in loop) and any(_loads(i) for i in loop) and (found is None or len(loop) < len(found))):
            found = loop
    return found


def _loads(instruction):
    return instruction.startswith("buffer_load") and instruction.endswith(" lds")


@pytest.mark.skipif(not os.path.exists(f"{LLVM}/llvm-objdump"), reason="no llvm-objdump")
def test_loads_ahead_of_the_matrix_instructions(tmp_path):
    link = tmp_path / "lib.so"
    link.symlink_to(_kernels.KERNEL_LIB_PATH)
    subprocess.run([f"{LLVM}/llvm-objdump", "--offloading", str(link)], check=True, cwd=tmp_path, stdout=subprocess.DEVNULL)
    forms = set()
    for code in tmp_path.glob("*gfx950"):
        symbols = subprocess.run([f"{LLVM}/llvm-objdump", "--syms", str(code)], check=True, text=True, stdout=subprocess.PIPE).stdout
        names = sorted({w for line in symbols.splitlines() for w in line.split()[-1:] if KERNEL.match(w)})
        if not names:
            continue
        listing = subprocess.run([f"{LLVM}/llvm-objdump", "-d", "--no-show-raw-insn", "--disassemble-symbols=" + ",".join(names), str(code)],
                                 check=True, text=True, stdout=subprocess.PIPE).stdout
        for part in re.split(r"^[0-9a-f]+ <", listing, flags=re.M)[1:]:
            name, _, text = part.partition(">:")
            loop = _k_loop(text.splitlines())
            assert loop, name
            assert [i for i in loop[:-1] if i.startswith(("s_branch", "s_cbranch"))] == [], name
            assert not any("saveexec" in i for i in loop), name
            kinds = ["load" if _loads(i) else "mfma" for i in loop if _loads(i) or i.startswith("v_mfma")]
            assert kinds == ["load", "mfma"] * (len(kinds) // 2), f"{name}: {kinds}"
            forms.add(KERNEL.match(name).groups())
    assert forms == {(t, k, l) for t in ("DF16_", "DF16b") for k in ("64", "128") for l in "123"}
