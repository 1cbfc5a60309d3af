"""Vector memory instructions written as assembly read only scalar registers that are safe to read: the compiler keeps five wait states between a
vector instruction's write of a scalar register (a buffer descriptor's words, by v_readfirstlane or out of a spill by v_readlane) and a vector memory
instruction that reads it, but does not look into assembly.  So a statement reads copies that scalar moves of its own made, or brings the five; and where it writes
m0, one instruction stands between that and the transfer that takes its LDS address from there."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "triton_amd", "csrc")
MEMORY = re.compile(r"(buffer|global|flat|scratch)_(load|store|atomic)")
STRING = r'"(?:[^"\\]|\\.)*"'
TOKEN = re.compile(rf"\s*(?:({STRING})|(\w+)|(\S))")


def _source(name):
    with open(os.path.join(CSRC, name)) as f:
        text = f.read().replace("\\\n", " ")
    return re.sub(rf"({STRING})|//[^\n]*", lambda m: m.group(1) or "", text)


def _macros(text):
    """name -> (parameters or None, body), of the macros whose body is one string literal after another (and macros)."""
    found = re.findall(r"#define (\w+)(?:\(([^)]*)\))?([^\n]*)", text)
    return {n: ([p.strip() for p in a.split(",")] if a else None, b.strip()) for n, a, b in found if re.fullmatch(rf"(?:{STRING}|\w+|\s|[(),])+", b.strip()) and '"' in b}


def _balanced(text, at):
    """The end of the parenthesis that opens at `at`."""
    depth = 0
    for m in re.finditer(rf"{STRING}|[()]", text[at:]):
        depth += {"(": 1, ")": -1}.get(m.group(), 0)
        if depth == 0:
            return at + m.end()
    raise AssertionError(f"no end of {text[at:at + 60]}")


def _expand(text, macros, used):
    """The string that a row of literals and macros makes, up to the first other token; the literals go into `used`."""
    out, at = "", 0
    while m := TOKEN.match(text, at):
        literal, name, other = m.groups()
        if literal:
            used.append(literal)
            out, at = out + literal[1:-1], m.end()
        elif name in ("R", "goto", "volatile", "inline"):
            at = m.end()
        elif name:
            params, body = macros[name]
            at = m.end()
            if params is not None:
                end = _balanced(text, text.index("(", at))
                args = [a.strip() for a in text[text.index("(", at) + 1:end - 1].split(",")]
                for p, a in zip(params, args, strict=True):
                    body = re.sub(rf"({STRING})|\b{p}\b", lambda m: m.group(1) or a, body)
                at = end
            out += _expand(body, macros, used)
        else:
            break
    return out


def _lines(whole):
    return [line.split() for line in re.split(r"(?:\\n|\\t|;)+", whole) if line.strip()]


def _statements(used=None):
    """Every assembly statement with a vector memory instruction, its macros expanded."""
    for name in sorted(os.listdir(CSRC)):
        if not name.endswith((".hip", ".h")):
            continue
        text = _source(name)
        macros = _macros(text)
        for m in re.finditer(r"\basm(?:\s+volatile)?\s*\(", text):
            literals = []
            lines = _lines(_expand(text[m.end():_balanced(text, m.end() - 1)], macros, literals))
            if any(MEMORY.match(line[0]) for line in lines):
                if used is not None:
                    used += [(name, s) for s in literals]
                yield name, lines


def safe(lines) -> bool:
    """Whether every vector memory instruction of a statement reads scalar registers of the statement's own making, or stands behind five wait states."""
    made, n, m0 = set(), 0, None
    for op, *args in lines:
        if MEMORY.match(op):
            named = re.findall(r"\bs(\d+|\[\d+:\d+\])", " ".join(args))
            if not (n >= 5 or (named and all(_range(r) <= made for r in named))) or (m0 is not None and n - m0 < 2 and "lds" in args):
                return False
        elif op.startswith("s_mov_b") and args[0].startswith("s"):
            made |= _range(args[0][1:].rstrip(","))
        elif op.startswith("v_read") and args[0].startswith("s"):
            return False  # (what this test is about, within one statement)
        if op.startswith("s_") and args and args[0] == "m0,":
            m0 = n
        n += int(args[0]) + 1 if op == "s_nop" else 1
    return True


def _range(r: str) -> set:
    a, b = r.strip("[]").split(":") if ":" in r else (r, r)
    return {f"s{i}" for i in range(int(a), int(b) + 1)}


def test_what_is_safe():
    load = ["buffer_load_dword", "%[o],", "s[4:7],", "0", "offen", "lds"]
    copies = [["s_mov_b64", "s[4:5],", "%[lo]"], ["s_mov_b64", "s[6:7],", "%[hi]"]]
    assert not safe([["s_nop", "0"], ["buffer_load_dword", "%0,", "%1,", "0"]])
    assert safe([["s_nop", "3"], ["s_mov_b32", "exec_hi,", "0"], ["buffer_load_dwordx4", "%0,", "%1,", "0"]])
    assert safe([*copies, load])
    assert not safe([copies[0], load])
    assert not safe([*copies, load, ["buffer_load_dword", "%[o],", "%[desc],", "0", "offen", "lds"]])  # a later one counts as well
    assert not safe([*copies, load, ["s_add_u32", "m0,", "m0,", "0x1000"], load])
    assert safe([*copies, load, ["s_add_u32", "m0,", "m0,", "0x1000"], *copies, load])


def test_macros_are_expanded():
    macros = _macros('#define A "x y\\n\\t"\n#define B(k) "z" k " w"\n#define C int\n')
    used = []
    assert _lines(_expand('A B(" u") "end" :: "s"(1)', macros, used)) == [["x", "y"], ["z", "u", "wend"]] and len(used) == 5


@pytest.mark.parametrize("name, lines", list(_statements()), ids=lambda v: v if isinstance(v, str) else v[-1][0])
def test_memory_instructions_in_assembly_read_settled_registers(name, lines):
    assert safe(lines), (name, lines)


def test_no_memory_instruction_is_missed():
    """Every string literal with a vector memory instruction, wherever it stands in the sources, belongs to a statement that was looked at."""
    used = []
    statements = list(_statements(used))
    for name in sorted(os.listdir(CSRC)):
        if name.endswith((".hip", ".h")):
            for literal in re.findall(STRING, _source(name)):
                assert not MEMORY.search(literal) or (name, literal) in used, (name, literal)
    assert sum(len([1 for line in lines if MEMORY.match(line[0])]) for _, lines in statements) >= 15
