"""Waits that the matrix cores' instructions are owed, in the kernels as they were built.

The hardware does not hold a matrix instruction back until an ordinary vector instruction before it has written its sources, nor an ordinary one
until a matrix instruction has written the result it wants: the program keeps them apart.  The compiler does that for the instructions that it
picks itself and does not look into written-out assembly, so the built code is read: every v_mfma's sources and the instructions up to two wait
states in front of it, along every way that leads there; and, in the kernels that write one out (`gemm_fourwave_kernel`), every result and what follows it
within the result's own time (the CDNA instruction set's table of required software waits: 2 after a vector write, passes + 3 after a
product of so many passes)."""
import os
import re
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from llm_rs_amd.csrc import build as native

AFTER_VECTOR_WRITE = 2
WRITTEN_OUT, AFTER_PRODUCT = "gemm_fourwave_kernel", {"v_mfma_f32_16x16x32_bf16": 4 + 3}        # (16 cycles: passes of four)
REGISTERS = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)")
BRANCH = re.compile(r"^s_c?branch\w*")


def registers(text):
    """The vector and accumulation registers that an operand names."""
    out = set()
    for bank, first, last, one in REGISTERS.findall(text):
        out.update((bank, r) for r in (range(int(first), int(last) + 1) if first else (int(one),)))
    return out


class Kernel:
    def __init__(self, name):
        self.name, self.ops, self.args, self.at = name, [], [], []

    def close(self, targets):
        """`targets`: address -> index of the code object's instructions that branches go to."""
        n = len(self.ops)
        place = {a: i for i, a in enumerate(self.at)}
        self.before, self.after = [[] for _ in range(n)], [[] for _ in range(n)]
        for i, op in enumerate(self.ops):
            goes = [] if op in ("s_endpgm", "s_branch") or i + 1 == n else [i + 1]
            if i in targets and targets[i] in place:
                goes.append(place[targets[i]])
            for j in goes:
                self.after[i].append(j)
                self.before[j].append(i)

    def waits(self, i):
        return int(self.args[i][0], 0) + 1 if self.ops[i] == "s_nop" else 1

    def within(self, i, states, ways):
        """The instructions fewer than `states` wait states away from i along `ways` (their index, once each)."""
        left, todo = {}, [(j, states) for j in ways[i]]
        while todo:
            j, s = todo.pop()
            if s <= 0 or left.get(j, 0) >= s:
                continue
            left[j] = s
            todo += [(k, s - self.waits(j)) for k in ways[j]]
        return left


def kernels_of(listing):
    """The kernels of a disassembled code object."""
    kernel, targets, start = None, {}, 0
    for line in listing.splitlines():
        if line.endswith(">:") and not line.startswith("\t"):
            if kernel is not None:
                kernel.close(targets)
                yield kernel
            kernel, targets, start = Kernel(line.split("<", 1)[1][:-2]), {}, int(line.split()[0], 16)
        elif line.startswith("\t") and "//" in line and kernel is not None:
            code, _, where = line.partition("//")
            op, _, args = code.strip().partition(" ")
            if BRANCH.match(op) and "+0x" in where:
                targets[len(kernel.ops)] = start + int(where.rsplit("+0x", 1)[1].rstrip("> "), 16)
            elif BRANCH.match(op) and where.rstrip().endswith(">"):
                targets[len(kernel.ops)] = start
            kernel.ops.append(re.sub(r"_(e32|e64|dpp|sdwa)$", "", op))
            kernel.args.append([a.strip() for a in re.split(r",(?![^\[]*\])", args)] if args.strip() else [])
            kernel.at.append(int(where.split(":")[0], 16))
    if kernel is not None:
        kernel.close(targets)
        yield kernel


def vector_writes(op, args):
    if not op.startswith("v_") or op.startswith("v_mfma") or op.startswith(("v_cmp", "v_readlane", "v_readfirstlane", "v_nop")):
        return set()
    return registers(" ".join(args[:2] if "swap" in op else args[:1]))


def faults_of(listing):
    faults = []
    for k in kernels_of(listing):
        for i, op in enumerate(k.ops):
            if not op.startswith("v_mfma"):
                continue
            wanted, result = registers(" ".join(k.args[i][1:4])), registers(k.args[i][0])
            for j in k.within(i, AFTER_VECTOR_WRITE, k.before):
                if vector_writes(k.ops[j], k.args[j]) & wanted:
                    faults.append(f"{k.name}: {k.ops[j]} {', '.join(k.args[j])} -> {op} {', '.join(k.args[i])}")
            for j in k.within(i, AFTER_PRODUCT.get(op, 0) if WRITTEN_OUT in k.name else 0, k.after):
                if not k.ops[j].startswith(("v_mfma", "s_")) and registers(" ".join(k.args[j])) & result:
                    faults.append(f"{k.name}: {op} {', '.join(k.args[i])} -> {k.ops[j]} {', '.join(k.args[j])}")
    return faults


SMALL = """
0000000000001000 <gemm_fourwave_kernel>:
\tv_mov_b32_e32 v5, v2                                       // 000000001000: 7E0A0302
\ts_waitcnt vmcnt(8)                                         // 000000001004: BF8C0F78
\tv_mfma_f32_16x16x32_bf16 v[2:5], v[10:13], v[14:17], v[2:5]// 000000001008: D3B50002 040A1D0A
\ts_nop 5                                                    // 000000001010: BF800005
\tv_add_f32_e32 v20, v3, v3                                  // 000000001014: 02280703
\ts_cbranch_scc1 65533                                       // 000000001018: BF85FFFB <gemm_fourwave_kernel+0x8>
\tv_mov_b32_e32 v10, 0                                       // 00000000101C: 7E140280
\ts_nop 0                                                    // 000000001020: BF800000
\ts_nop 0                                                    // 000000001024: BF800000
\ts_branch 65528                                             // 000000001028: BF82FFF8 <gemm_fourwave_kernel+0x8>
"""


def test_the_reading_itself():
    """A write one state before its product, a result read one too early, and a write that a branch brings three states before."""
    assert [f.split(" -> ")[0].split(": ")[1].split()[0] for f in faults_of(SMALL)] == ["v_mov_b32", "v_mfma_f32_16x16x32_bf16"]
    assert len(faults_of(SMALL.replace("s_nop 5", "s_nop 6"))) == 1
    assert len(faults_of(SMALL.replace("s_waitcnt vmcnt(8) ", "s_nop 1").replace("s_nop 5", "s_nop 6"))) == 0
    assert len(faults_of(SMALL.replace("\ts_nop 0  ", "\tv_nop    ").replace("s_nop 5", "s_nop 6"))) == 1


def test_every_matrix_instruction_has_its_waits(tmp_path):
    objdump = shutil.which("llvm-objdump", path="/opt/rocm/llvm/bin" + os.pathsep + os.environ.get("PATH", ""))
    if objdump is None:
        pytest.skip("no llvm-objdump to read the built kernels with")
    library = str(tmp_path / "kernels.so")
    shutil.copy(native.build_hip(), library)
    subprocess.run([objdump, "--offloading", library], check=True, capture_output=True, cwd=tmp_path)
    objects = sorted(str(tmp_path / f) for f in os.listdir(tmp_path) if native.GPU_ARCH in f)
    assert objects
    dump = lambda path: subprocess.run([objdump, "-d", "--no-show-raw-insn", path], check=True, capture_output=True, text=True).stdout
    with ThreadPoolExecutor(4) as pool:
        listings = list(pool.map(dump, objects))
    assert sum(text.count("v_mfma") for text in listings) > 1000
    faults = [f for text in listings if "v_mfma" in text for f in faults_of(text)]
    assert not faults, f"{len(faults)} waits too short:\n" + "\n".join(faults[:40])
