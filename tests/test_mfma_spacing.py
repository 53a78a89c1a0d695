"""The built kernels' wait states between matrix instructions and what touches their results.

The hardware does not hold a VALU or memory instruction back until a matrix instruction's result
has arrived; the compiler spaces the two, but not for instructions inside inline assembly
(csrc/mfma.hpp, settle()). This looks through libie_hip.so's gfx950 instructions, along every
path, for one that reads or overwrites a result register too early. No GPU needed."""
from __future__ import annotations

import collections
import os
import re
import shutil
import subprocess

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
# Wait states until a result may be read or overwritten, as the compiler places them (s_nop 7
# and s_nop 9 in `c = mfma(..); x = c[0] + c[1]`).
WAIT = {"v_mfma_f32_16x16x32_bf16": 8, "v_mfma_f32_16x16x32_f16": 8, "v_mfma_f32_16x16x4_f32": 10}
REGISTERS = re.compile(r"\bv(?:\[(\d+):(\d+)\]|(\d+))")


def registers(text):
    out = set()
    for lo, hi, one in REGISTERS.findall(text):
        out.update(range(int(lo), int(hi) + 1) if lo else [int(one)])
    return out


def functions(listing):
    """(name, [(address, mnemonic, operands, branch target or None)]) of a disassembly."""
    name, body = None, []
    for line in listing.splitlines():
        head = re.match(r"^([0-9a-f]+) <(.+)>:$", line)
        if head:
            if name:
                yield name, body
            name, body, start = head[2], [], int(head[1], 16)
            continue
        code = re.match(r"^\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+):?(.*)$", line)
        if code and name:
            to = re.search(r"<.*\+0x([0-9a-f]+)>", code[2] + code[4])
            body.append((int(code[3], 16), code[1], code[2], start + int(to[1], 16) if to else None))
    if name:
        yield name, body


def too_early(body):
    """Indexes of instructions that touch a matrix result before it has arrived."""
    at = {ins[0]: i for i, ins in enumerate(body)}
    pending = [None] * len(body)  # on entry: wait states left per register, the worst over paths
    pending[0] = {}
    bad, work = set(), collections.deque([0])
    while work:
        i = work.popleft()
        _, op, args, target = body[i]
        mfma = op.startswith("v_mfma")
        if not mfma and op[:2] in ("v_", "ds", "gl", "bu", "fl", "sc"):
            if any(pending[i].get(r, 0) > 0 for r in registers(args)):
                bad.add(i)
        states = 1 + int(args) if op == "s_nop" else 1
        after = {r: n - states for r, n in pending[i].items() if n > states}
        if mfma:
            after.update(dict.fromkeys(registers(args.split(", ")[0]), WAIT[op]))
        follow = [] if op in ("s_endpgm", "s_branch") else [i + 1]
        if op.startswith(("s_branch", "s_cbranch")):
            follow.append(at[target])
        for j in follow:
            if j >= len(body):
                continue
            known = pending[j]
            if known is None:
                pending[j] = dict(after)
                work.append(j)
            elif any(n > known.get(r, 0) for r, n in after.items()):
                for r, n in after.items():
                    known[r] = max(n, known.get(r, 0))
                work.append(j)
    return sorted(bad)


def test_finds_an_early_read():
    """Seven wait states, along a taken branch, are one too few; eight are enough; a register
    of the result that is overwritten counts as one that is read."""
    def body(nops, last):
        ops = [("v_mfma_f32_16x16x32_f16", "v[4:7], v[8:11], v[12:15], 0", None),
               ("s_cbranch_scc1", "2", 12), ("s_endpgm", "", None),
               ("s_nop", str(nops - 2), None), ("v_max_f32_e32", last, None), ("s_endpgm", "", None)]
        return [(4 * i, *o) for i, o in enumerate(ops)]
    assert too_early(body(7, "v0, v1, v6")) == [4]
    assert too_early(body(7, "v5, v1, v2")) == [4]
    assert too_early(body(7, "v0, v1, v8")) == []
    assert too_early(body(8, "v0, v1, v6")) == []


def test_built_kernels(ie, tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    lib = shutil.copy(ie.LIB_PATH, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True)
    seen, bad = 0, []
    for part in sorted(tmp_path.glob("*amdgcn*")):
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", part], check=True,
                              capture_output=True, text=True).stdout
        for name, body in functions(text):
            seen += sum(op.startswith("v_mfma") for _, op, *_ in body)
            bad += [f"{name}+{body[i][0] - body[0][0]:#x}: {body[i][1]} {body[i][2]}"
                    for i in too_early(body)]
    assert seen > 1000 and not bad, "\n".join(bad)
