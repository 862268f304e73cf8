"""The inline assembly of the path layout (csrc/g1_path.h) in the code that the library's flags give. The compiler counts
the wait states between its own instructions and none across an inline assembly block, so a block holds those that its
reads need whatever the compiler puts in front of it (a register copy, a spilled value's reload), and its results are
not read too early after it. On gfx950: two between a vector instruction's write of a register and a read by DPP or a
lane swap, one before a v_readlane, one after a transcendental, two from a vector instruction's write of a scalar
register to a vector instruction's read. CPU only: compiles to assembly."""
import os
import re
import subprocess

import pytest

from nablaengine_amd import build

TRANS = re.compile(r"v_(rsq|rcp|sqrt|exp|log|sin|cos)_")


def _regs(x):
    r = set(re.findall(r"\b[vs]\d+\b", x))
    for k, a, b in re.findall(r"\b([vs])\[(\d+):(\d+)\]", x):
        r |= {f"{k}{i}" for i in range(int(a), int(b) + 1)}
    return r


def _instructions(text):
    """(instruction, number of its inline assembly block or 0) in program order."""
    block = inside = 0
    for line in text.splitlines():
        s = line.split(";")[0].strip() if ";;#" not in line else line.strip()
        if s.startswith(";;#ASMSTART"):
            block, inside = block + 1, 1
        elif s.startswith(";;#ASMEND"):
            inside = 0
        elif re.match(r"(v|s|ds|global|scratch|buffer|flat)_\w+", s):
            yield s, block * inside


@pytest.mark.parametrize("source", ["g1_forward.hip", "g1_adjoint.hip"])
def test_each_assembly_block_holds_its_wait_states(source, tmp_path):
    out = tmp_path / "a.s"
    flags = [f for f in build.FLAGS if f not in ("-fPIC", "-shared")]
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    subprocess.run([hipcc, *flags, "--cuda-device-only", "-S", "-o", str(out), os.path.join(build.CSRC, source)],
                   check=True, capture_output=True)
    t = seen = last = start = 0
    wrote = {}  # register -> (time, block, transcendental) of the last vector instruction that wrote it
    for ins, block in _instructions(out.read_text()):
        if block != last:
            start, last = t, block
        op, _, rest = ins.partition(" ")
        if op == "s_nop":
            t += int(rest) + 1
            continue
        ops = [x.strip() for x in rest.split(",")]
        if op.startswith("v_"):
            swap, dpp = "permlane" in op, "_dpp" in op
            if dpp and block:
                seen += 1
                # what the block reads by DPP was written in it, or might have been written right before it
                for r in _regs(ops[1]):
                    w = wrote.get(r)
                    assert t - (w[0] + 1 if w and w[1] == block else start) >= 2, (ins, "opens too early")
            for i, x in enumerate(ops):
                for r in _regs(x):
                    w = wrote.get(r)
                    if not w or (not block and not w[1]) or (i == 0 and not swap):
                        continue  # the compiler's own pair, or the result
                    need = 2 if swap or r[0] == "s" or (dpp and i == 1) else 1 if w[2] or op.startswith("v_readlane") else 0
                    assert t - w[0] - 1 >= need, (ins, r, t, w)
            for r in _regs(ops[0]) | (_regs(ops[1]) if swap else set()):
                wrote[r] = (t, block, bool(TRANS.match(op)))
        t += 1
    assert seen > 200, seen
