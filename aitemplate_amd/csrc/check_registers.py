"""Build-time check of the kernels whose instructions the compiler does not wait for by itself.

gemm_kernel_wide.hpp and gemm_kernel_rows.hpp read LDS, and the former multiplies, through inline asm.  The compiler takes an
asm's outputs for there at once: nothing in the source keeps it from placing a copy or a spill of one between the read and the
wait behind it, and it would take the register's old contents.  So the code of every such kernel in an object is followed here
along all its paths:

* a register that an LDS read fills is named by no other instruction until a wait has it arrived;
* in the wide kernel, a register that a matrix instruction writes is named by no other kind of instruction for WAIT_STATES
  issue slots (where the multiplications are the compiler's own it counts the slots itself).

    python3 check_registers.py object.o ...     (exits with 1 and says where, if a kernel does otherwise)
"""
import os
import re
import subprocess
import sys
import tempfile

KERNELS = re.compile(r"gemm_rcr_(wide|rows)_kernel")
MULTIPLY = re.compile(r"gemm_rcr_wide_kernel")  # ... of which these through asm
WAIT_STATES = 19  # the most that the results of a matrix instruction take (16 passes) until others may read them
LLVM = os.environ.get("ROCM_LLVM_BIN", "/opt/rocm/llvm/bin")

_REG = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)")
_LINE = re.compile(r"^\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+):(.*)$")
_SYMBOL = re.compile(r"^([0-9a-f]+) <(.*)>:$")
_TARGET = re.compile(r"<(.*?)(?:\+0x([0-9a-f]+))?>")


class Instruction:
    def __init__(self, address, op, operands, target):
        self.address, self.op, self.operands, self.target = address, op, operands, target
        named = []
        for m in _REG.finditer(operands):
            first, last = (m[2], m[3]) if m[2] else (m[4], m[4])
            named.append(frozenset((m[1], i) for i in range(int(first), int(last) + 1)))
        self.named = frozenset().union(*named)
        self.first = named[0] if named else frozenset()
        self.reads_lds = op.startswith("ds_read")
        self.counts_lgkm = op.startswith(("ds_", "s_load", "s_buffer_load"))
        self.multiplies = op.startswith("v_mfma")
        self.branches = op == "s_branch" or op.startswith("s_cbranch")
        self.falls_through = op not in ("s_branch", "s_endpgm")
        self.slots = int(operands, 0) + 1 if op == "s_nop" else 1
        m = re.search(r"lgkmcnt\((\d+)\)", operands) if op == "s_waitcnt" else None
        self.waits_to = int(m[1]) if m else None


def parse(listing):
    """{kernel: [Instruction]} of llvm-objdump's listing, the kernels that KERNELS names."""
    kernels, body, symbol, start = {}, None, None, 0
    for line in listing.splitlines():
        m = _SYMBOL.match(line)
        if m:
            symbol, start = m[2], int(m[1], 16)
            body = kernels.setdefault(symbol, []) if KERNELS.search(symbol) else None
            continue
        m = _LINE.match(line) if body is not None else None
        if m:
            target = None
            if m[1].startswith(("s_branch", "s_cbranch")):
                t = _TARGET.search(m[4])
                if t is None or t[1] != symbol:
                    raise ValueError(f"{symbol}: branch out of the kernel at {m[3]}")
                target = start + int(t[2] or "0", 16)
            elif m[1].startswith(("s_setpc", "s_swappc", "s_call", "s_cbranch_i_fork", "s_cbranch_g_fork", "s_cbranch_join")):
                raise ValueError(f"{symbol}: {m[1]} at {m[3]} is not followed")
            body.append(Instruction(int(m[3], 16), m[1], m[2], target))
    return kernels


def _step(ins, state, report):
    """The state behind an instruction: (register -> lgkm operations issued since its read, at least; register -> issue slots since
    the matrix instruction that writes it, at least)."""
    pending, results = state
    for reg in ins.named & pending.keys():
        report(ins, reg, "an LDS read that has not arrived")
    if not ins.multiplies:
        for reg in ins.named & results.keys():
            report(ins, reg, f"a matrix instruction {results[reg]} issue slots before")
    if ins.waits_to is not None:
        pending = {reg: n for reg, n in pending.items() if n < ins.waits_to}
    if ins.counts_lgkm:
        pending = {reg: n + 1 for reg, n in pending.items()}
        if ins.reads_lds:
            pending.update((reg, 0) for reg in ins.first)
    results = {reg: n + ins.slots for reg, n in results.items() if n + ins.slots < WAIT_STATES}
    if ins.multiplies:
        results.update((reg, 0) for reg in ins.first)
    return pending, results


def check(body, multiplies=True):
    """What a kernel does wrong, as texts; `multiplies`: through asm."""
    at = {ins.address: i for i, ins in enumerate(body)}
    faults = {}

    def report(ins, reg, what):
        faults[(ins.address, reg)] = f"{ins.address:x}: {ins.op} {ins.operands} names {reg[0]}{reg[1]} of {what}"

    starts = {0} | {at[ins.target] for ins in body if ins.branches} | {i + 1 for i, ins in enumerate(body) if ins.branches}
    entry, todo = {0: ({}, {})}, [0]
    while todo:
        i = todo.pop()
        state = entry[i]
        while True:
            ins = body[i]
            state = _step(ins, state, report)
            if not multiplies:
                state = state[0], {}
            nexts = [at[ins.target]] if ins.branches else []
            i += 1
            if ins.falls_through and i < len(body):
                if i not in starts and not nexts:
                    continue
                nexts.append(i)
            break
        for n in nexts:
            merged = state
            if n in entry:  # the fewest operations and slots over the paths that lead here
                merged = tuple({r: min(a.get(r, 1 << 30), b.get(r, 1 << 30)) for r in a.keys() | b.keys()} for a, b in zip(entry[n], state))
                if merged == entry[n]:
                    continue
            entry[n] = merged
            todo.append(n)
    return list(faults.values())


def listing_of(path):
    """llvm-objdump's listing of the kernels in an object with one gfx950 code object in it."""
    with tempfile.TemporaryDirectory() as d:
        link = os.path.join(d, "o.o")
        os.symlink(os.path.abspath(path), link)
        subprocess.run([f"{LLVM}/llvm-objdump", "--offloading", link], check=True, cwd=d, stdout=subprocess.DEVNULL)
        code = [f for f in os.listdir(d) if f.endswith("gfx950")]
        if len(code) != 1:
            raise ValueError(f"{path}: no code object for gfx950 found")
        code = os.path.join(d, code[0])
        names = subprocess.run([f"{LLVM}/llvm-objdump", "--syms", code], check=True, text=True, stdout=subprocess.PIPE).stdout
        wanted = sorted({w for line in names.splitlines() for w in line.split()[-1:] if KERNELS.search(w) and "." not in w})
        if not wanted:
            return ""
        return subprocess.run([f"{LLVM}/llvm-objdump", "-d", "--no-show-raw-insn", "--disassemble-symbols=" + ",".join(wanted), code],
                              check=True, text=True, stdout=subprocess.PIPE).stdout


def main(paths):
    bad = 0
    for path in paths:
        for symbol, body in parse(listing_of(path)).items():
            faults = check(body, bool(MULTIPLY.search(symbol)))
            bad += len(faults)
            for fault in faults[:8]:
                print(f"{path}: {symbol}: {fault}", file=sys.stderr)
    return 1 if bad else 0


if __name__ == "__main__":
    sys.exit(main(sys.argv[1:]))
