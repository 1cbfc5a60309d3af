"""Vector memory instructions written as assembly read only scalar registers that are safe to read: the compiler keeps five wait states between a
vector instruction's write of a scalar register (a buffer descriptor's words, by v_readfirstlane or out of a spill by v_readlane) and a vector memory
instruction that reads it, but does not look into assembly.  So a statement reads copies that scalar moves of its own made, or brings the five."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "triton_amd", "csrc")
MEMORY = re.compile(r"(buffer|global|flat|scratch)_")


def _statements():
    for name in sorted(os.listdir(CSRC)):
        if name.endswith((".hip", ".h")):
            with open(os.path.join(CSRC, name)) as f:
                text = f.read()
            macros = dict(re.findall(r'#define (\w+) "((?:[^"\\]|\\.)*)"', text))
            for m in re.finditer(r'asm(?:\s+volatile)?\s*\(\s*((?:\w+\s+)?)"((?:[^"\\]|\\.)*)"', text):
                whole = macros.get(m.group(1).strip(), "") + m.group(2)
                lines = [line.split() for line in re.split(r"\\n(?:\\t)?", whole) if line.strip()]
                if any(MEMORY.match(line[0]) for line in lines):
                    yield name, lines


def safe(lines) -> bool:
    """Whether the statement's first vector memory instruction reads scalar registers of the statement's own making, or stands behind five wait states."""
    made, n = set(), 0
    for op, *args in lines:
        if MEMORY.match(op):
            named = re.findall(r"\bs(\d+|\[\d+:\d+\])", " ".join(args))
            return n >= 5 or (bool(named) and all(_range(r) <= made for r in named))
        if op.startswith("s_mov_b") and args[0].startswith("s"):
            made |= _range(args[0][1:].rstrip(","))
        n += int(args[0]) + 1 if op == "s_nop" else 1
    return True


def _range(r: str) -> set:
    a, b = r.strip("[]").split(":") if ":" in r else (r, r)
    return {f"s{i}" for i in range(int(a), int(b) + 1)}


def test_what_is_safe():
    load = ["buffer_load_dword", "%[o],", "s[4:7],", "0", "offen", "lds"]
    assert not safe([["s_nop", "0"], ["buffer_load_dword", "%0,", "%1,", "0"]])
    assert safe([["s_nop", "3"], ["s_mov_b32", "exec_hi,", "0"], ["buffer_load_dwordx4", "%0,", "%1,", "0"]])
    assert safe([["s_mov_b64", "s[4:5],", "%[lo]"], ["s_mov_b64", "s[6:7],", "%[hi]"], load])
    assert not safe([["s_mov_b64", "s[4:5],", "%[lo]"], load])


@pytest.mark.parametrize("name, lines", list(_statements()), ids=lambda v: v if isinstance(v, str) else v[-1][0])
def test_memory_instructions_in_assembly_read_settled_registers(name, lines):
    assert safe(lines), (name, lines)


def test_there_are_such_statements():
    assert len(list(_statements())) >= 5
