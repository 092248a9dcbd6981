"""What the build looks for in the device assembly of a unit: copies to the LDS whose hazards nobody else looks after.

Kernels that transpose an operand as they read it issue their copies (``buffer_load ... lds``) in ``asm`` statements, which
the compiler's hazard recognizer does not look into. A load must be five wait states behind a VALU instruction that wrote a
scalar register of its descriptor (``v_readfirstlane``, ``v_readlane`` of a spilled one), and M0, which names the
place in the LDS, must be written by these statements alone. Waiting in every statement instead costs the
products that copy both operands so 3.5 % (8192 x 8192 x 2048 101.3 -> 105.0 us)."""

from __future__ import annotations

import re

WAIT_STATES = 5


def functions(lines):
    """``(name, first line, last line)`` of each function."""
    cur = None
    for i, line in enumerate(lines):
        m = re.match(r"^(_Z\w+):", line)
        if m:
            cur = (m.group(1), i)
        elif cur is not None and line.startswith(".Lfunc_end"):
            yield (*cur, i)
            cur = None


def _scalars(operand: str) -> set[int]:
    m = re.fullmatch(r"s(?:(\d+)|\[(\d+):(\d+)\])", operand)
    if m is None:
        return set()
    return {int(m[1])} if m[1] else set(range(int(m[2]), int(m[3]) + 1))


def _written_by_valu(op: str, operands: list[str]) -> set[int]:
    if not op.startswith("v_"):
        return set()
    carries = re.search(r"_co_|div_scale|mad_[iu]64", op) is not None  # (a second, scalar result)
    return set().union(*map(_scalars, operands[:2 if carries else 1]))


def faults_of_copies(body) -> tuple[int, list[str]]:
    """``(copies, faults)`` of a function's lines: how many copies to the LDS it has in ``asm`` statements, and what is wrong with
    them or, as to the wait states, with any such copy."""
    code, in_asm, inside = [], [], False
    for x in body:
        if "#ASMSTART" in x or "#ASMEND" in x:
            inside = "#ASMSTART" in x
        x = x.split(";")[0].strip()
        if x and (not x.startswith(".") or x.endswith(":")):
            code.append((x, *x.replace(",", " ").split()))
            in_asm.append(inside)
    jumps: dict[str, list[int]] = {}
    for i, (x, op, *operands) in enumerate(code):
        if op.startswith(("s_branch", "s_cbranch")):
            jumps.setdefault(operands[0], []).append(i)

    def written(i: int, states: int, registers: set[int]) -> bool:
        """Whether one of the last ``states`` wait states in front of line ``i``, on any way to it, is a VALU write."""
        while states > 0 and i > 0:
            i -= 1
            x, op, *operands = code[i]
            if x.endswith(":"):
                if any(written(j, states - 1, registers) for j in jumps.get(x[:-1], ())):
                    return True
                continue
            if op in ("s_branch", "s_endpgm", "s_setpc_b64"):
                return False
            if _written_by_valu(op, operands) & registers:
                return True
            states -= int(operands[0], 0) + 1 if op == "s_nop" else 1
        return False

    copies, faults = 0, []
    for i, (x, op, *operands) in enumerate(code):
        if re.match(r"buffer_load_\w+ .*\blds\b", x):
            copies += in_asm[i]
            if written(i, WAIT_STATES, next(s for o in operands if len(s := _scalars(o)) == 4)):
                faults.append(f"less than {WAIT_STATES} wait states from a VALU write of the descriptor: {x}")
    if copies:
        faults += [f"M0 is used besides the copies: {x}" for i, (x, *_) in enumerate(code) if not in_asm[i] and re.search(r"\bm0\b", x)]
    return copies, faults


def check(lines, what: str) -> int:
    """Copies in ``asm`` statements of a unit's assembly; raises where one is not safe."""
    total = 0
    for name, first, last in functions(lines):
        copies, faults = faults_of_copies(lines[first:last])
        total += copies
        if faults:
            raise RuntimeError(f"{what}: {name}: {len(faults)} unsafe uses, the first: {faults[0]}")
    return total
