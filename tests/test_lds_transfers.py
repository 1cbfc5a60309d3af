"""Vector memory instructions written as assembly bring the wait states that the compiler keeps only for its own: five between a vector instruction's
write of a scalar register (a buffer descriptor's words, by v_readfirstlane or out of a spill by v_readlane) and a vector memory instruction that reads it."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "triton_amd", "csrc")


def _statements():
    for name in sorted(os.listdir(CSRC)):
        if name.endswith((".hip", ".h")):
            with open(os.path.join(CSRC, name)) as f:
                text = f.read()
            for m in re.finditer(r'asm(?:\s+volatile)?\s*\(\s*"((?:[^"\\]|\\.)*)"', text):
                lines = [line.split() for line in re.split(r"\\n(?:\\t)?", m.group(1)) if line.strip()]
                if any(re.match(r"(buffer|global|flat|scratch)_", line[0]) for line in lines):
                    yield name, lines


def wait_states(lines) -> int:
    """Wait states that the statement itself puts in front of its first vector memory instruction."""
    n = 0
    for op, *args in lines:
        if re.match(r"(buffer|global|flat|scratch)_", op):
            return n
        n += int(args[0]) + 1 if op == "s_nop" else 1
    return n


def test_wait_states_are_counted():
    assert wait_states([["s_nop", "0"], ["buffer_load_dword", "v0"]]) == 1
    assert wait_states([["s_nop", "3"], ["s_mov_b32", "exec_hi,", "0"], ["buffer_load_dwordx4", "v0"]]) == 5


@pytest.mark.parametrize("name, lines", list(_statements()), ids=lambda v: v if isinstance(v, str) else v[-1][0])
def test_memory_instructions_in_assembly_bring_their_wait_states(name, lines):
    assert wait_states(lines) >= 5, (name, lines)


def test_there_are_such_statements():
    assert len(list(_statements())) >= 5
