"""A scalar register that a vector instruction wrote (a reload of a spilled one among them) may be read by a vector-memory
instruction five wait states later at the earliest. The compiler keeps that distance for its own instructions and does not look
into assembly statements: those with vector-memory instructions on scalar operands have to bring it along."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vllm-kunlun_amd", "csrc")
DISTANCE = 5


def _statements():
    """(file and line, instructions, scalar inputs) of every assembly statement with a vector-memory instruction."""
    for path in sorted(glob.glob(os.path.join(CSRC, "*"))):
        text = open(path).read()
        for m in re.finditer(r"\basm\s*(?:volatile)?\s*\(", text):
            depth, end = 1, m.end()
            while depth:  # (no parenthesis stands inside the statements' strings)
                depth += {"(": 1, ")": -1}.get(text[end], 0)
                end += 1
            body = text[m.end():end - 1]
            code, *operands = re.split(r"(?<=\")\s*\n?\s*:", body, maxsplit=1)
            lines = [s.strip() for s in "".join(re.findall(r'"([^"]*)"', code)).replace("\\t", "").split("\\n") if s.strip()]
            if any(s.startswith(("buffer_", "global_")) for s in lines):
                scalars = re.findall(r'\[(\w+)\]\s*"\+?=?&?s"', operands[0])
                yield f"{os.path.basename(path)}:{text.count(chr(10), 0, m.start()) + 1}", lines, scalars


def _shortest(lines, scalars):
    """Wait states between the statement's start and each use of a scalar operand by a vector-memory instruction, at least."""
    at = {}
    for i, s in enumerate(lines):
        if re.fullmatch(r"\d+:", s):
            at[s[:-1]] = i
    best, todo, found = {}, [(0, 0)], []
    while todo:
        i, n = todo.pop()
        if i >= len(lines) or best.get(i, 1 << 30) <= n:
            continue
        best[i] = n
        op, *rest = lines[i].split(None, 1)
        args = rest[0] if rest else ""
        if op.startswith(("buffer_", "global_")) and any(f"%[{r}]" in args for r in scalars):
            found.append(n)
        step = 0 if op.endswith(":") else int(args) + 1 if op == "s_nop" else 1
        if op.startswith(("s_branch", "s_cbranch")):
            todo.append((at[args[:-1]], n + 1))
        if op != "s_branch":
            todo.append((i + 1, n + step))
    return min(found, default=None)


STATEMENTS = list(_statements())


def test_statements_are_found():
    assert {where.split(":")[0] for where, _, _ in STATEMENTS} == {"macro_tile.hip", "tiled_gemm.hip"}


@pytest.mark.parametrize("where,lines,scalars", STATEMENTS, ids=[s[0] for s in STATEMENTS])
def test_distance(where, lines, scalars):
    assert scalars and _shortest(lines, scalars) >= DISTANCE, lines
