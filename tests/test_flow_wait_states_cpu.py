"""Wait states in front of the multiply-adds with a broadcast inside
(chol_flow.hip: fma_row_lane).  Their DPP operand is inside inline assembly, so
the compiler inserts no wait states: two must lie between a vector instruction
that writes the register and the multiply-add that reads it across lanes, and
five after one that writes EXEC.  A copy that the register allocator puts in
front of one would break that in the generated code only, so this looks there."""
from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "exageostat_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"
FMA = "v_fmac_f64_dpp"


def _regs(operand):
    """Vector registers of an operand: v7 or v[6:7], with or without a sign."""
    m = re.fullmatch(r"-?\|?v(?:(\d+)|\[(\d+):(\d+)\])\|?", operand)
    if not m:
        return set()
    if m.group(1):
        return {int(m.group(1))}
    return set(range(int(m.group(2)), int(m.group(3)) + 1))


def _hazards(lines):
    """(line number, text) of every FMA whose DPP operand may be written too
    late, and the number of FMAs."""
    code = []  # (opcode, operands) or (None, None) for a label
    bad, count = [], 0
    for number, line in enumerate(lines, 1):
        line = line.split(";")[0].strip()
        if not line or line.startswith("."):
            if re.fullmatch(r"\.LBB\w+:", line):
                code.append((None, None))
            continue
        if line.endswith(":"):
            code.append((None, None))
            continue
        op, _, rest = line.partition(" ")
        operands = [o.strip() for o in rest.split(",")]
        if op == FMA:
            count += 1
            source = _regs(operands[1].split(" ")[0])
            assert len(source) == 2, line
            states = 0
            for prev, ops in reversed(code):
                if states >= 5:
                    break
                if prev is None:  # a jump's target: what precedes is not known
                    if states < 2:
                        bad.append((number, line))
                    break
                if prev.startswith("v_cmpx"):
                    bad.append((number, line))
                    break
                # conservative: vector instructions write their first operand
                if states < 2 and prev.startswith("v_") and _regs(ops[0]) & source:
                    bad.append((number, line))
                    break
                states += int(ops[0], 0) + 1 if prev == "s_nop" else 1
        code.append((op, operands))
    return bad, count


def test_the_check_finds_hazards():
    late = ["v_mov_b32_e32 v4, v9", "s_nop 0", f"{FMA} v[0:1], v[4:5], v[2:3] row_newbcast:1 row_mask:0xf"]
    assert _hazards(late) == ([(3, late[2])], 1)
    assert _hazards([late[0], "s_nop 1", late[2]]) == ([], 1)
    assert _hazards([".LBB0_1:", "s_nop 0", late[2]])[0]
    assert _hazards(["v_cmpx_lt_i32_e32 v1, v2", "s_nop 3", late[2]])[0]
    assert not _hazards(["v_cmpx_lt_i32_e32 v1, v2", "s_nop 4", late[2]])[0]


@pytest.mark.skipif(not shutil.which(HIPCC), reason="needs hipcc")
def test_wait_states_in_the_generated_code(tmp_path):
    with open(os.path.join(ROOT, "exageostat_amd", "Makefile")) as f:
        flags = re.search(r"^CXXFLAGS = (.*?[^\\])\n", f.read(), re.M | re.S).group(1)
    flags = flags.replace("\\\n", " ").replace("$(ARCH)", "gfx950").split()
    out = tmp_path / "chol_flow.s"
    subprocess.run([HIPCC, *flags, "-S", "--cuda-device-only", os.path.join(CSRC, "chol_flow.hip"), "-o", str(out)],
                   check=True, capture_output=True)
    bad, count = _hazards(out.read_text().split("\n"))
    assert count > 0
    assert not bad, bad[:5]
