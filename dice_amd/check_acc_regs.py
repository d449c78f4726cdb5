"""Build-time check of the expert GEMM kernels whose sums live in accumulation
registers that only inline assembly names (csrc/grouped_gemm_persist.hip).

The compiler does not know that those registers are in use.  When it runs out
of vector registers it parks values in accumulation registers of its own
choice, lowest numbers first; a kernel of sixteen blocks owns all 256 and must
see none of that, a kernel of twelve blocks keeps its sums in a64 .. a255 and
leaves a0 .. a63 to the compiler.  A kernel whose k-loop is assembly text
(gemm_persist_kernel4a, gemm_persist_kernel_f8a) also names its register stages, v128 .. v255, in that
text only: it is compiled with a budget of 128 vector registers and must see
the compiler neither above v127 nor in any accumulation register
(gemm_persist_kernel_f8s: the text names v117 .. v127 as well).  This script
reads the device assembly the compiler wrote for a translation unit and fails
the build if an instruction outside the inline assembly touches a register that
belongs to the assembly.

Nor does the compiler know which LDS reads the assembly has left in flight.  The
staged kernels (fragments in v0 .. v63) leave a tile's last statement with reads of
the next tile's first fragments under way, and those that copy straight to LDS
(gemm_persist_kernel4d, gemm_persist_kernel_f8d: v0 .. v127) also run compiled
code - a whole tile switch - between the two statements of every step with those
of the second k-block under way.  A value moved out of such a register has not
arrived yet, one put there is overwritten when it does.  So every path from a
statement that reads fragments to the next statement that waits for all of LDS
(lgkmcnt(0)) is followed, and an instruction of the compiler on it that names a
fragment's register fails the build as well.  (Its own waits do not end a path:
the fragments are the assembly's for the whole k-loop.)
"""
from __future__ import annotations

import re
import sys

_KERNEL = re.compile(r"^(_ZN4dice\S*gemm_persist_kernel(?:4[ad]?|_f8[asd])I\S+):")
_ANY_FN = re.compile(r"^(\S+):\s*(;.*)?$")
_LABEL = re.compile(r"^(\.L\w+):")
_DRAINS = re.compile(r"^s_waitcnt\b.*\blgkmcnt\(0\)")
_REG = re.compile(r"\b([av])(\d+)\b|\b([av])\[(\d+):(\d+)\]")


def _owned_from(mangled: str):
    """(first accumulation register, first vector register) the assembly owns."""
    if "gemm_persist_kernel4aI" in mangled or "gemm_persist_kernel_f8aI" in mangled:
        return 0, 128
    if "gemm_persist_kernel4dI" in mangled or "gemm_persist_kernel_f8dI" in mangled:   # (no vector register is the text's for good)
        return 0, 256
    if "gemm_persist_kernel_f8sI" in mangled:     # the scaled kind's text also names v117 .. v127
        return 0, 117
    # gemm_persist_kernel4<MODE, HAS_BIAS, BN, ...>: ILi<mode>ELb<bias>ELi<BN>E...
    m = re.search(r"gemm_persist_kernel4ILi\d+ELb[01]ELi(\d+)E", mangled)
    if not m:
        raise RuntimeError(f"cannot read the tile width from {mangled}")
    return (0 if int(m.group(1)) == 256 else 64), 256


def _fragments_end(mangled: str) -> int:
    """The fragments that the assembly reads from LDS are the vector registers below this one (0: not checked)."""
    if re.search(r"gemm_persist_kernel(?:4d|_f8d)I", mangled):
        return 128
    return 64 if re.search(r"gemm_persist_kernel(?:4a|_f8a|_f8s)I", mangled) else 0


def _registers(code: str):
    """(file, first, last) of every accumulation or vector register that an instruction names."""
    for m in _REG.finditer(code):
        if m.group(1):
            yield m.group(1), int(m.group(2)), int(m.group(2))
        else:
            yield m.group(3), int(m.group(4)), int(m.group(5))


def _after_statement(lines):
    """Whether LDS reads may be in flight behind a statement of the assembly (None: it neither reads nor waits)."""
    in_flight = None
    for ln in lines:
        if ln.startswith("ds_read"):
            in_flight = True
        elif _DRAINS.match(ln):
            in_flight = False
    return in_flight


def _early_touches(body, fragments_end: int):
    """Instructions of the compiler that name a fragment's register between a statement that reads and one that waits.
    `body`: ("label", name), ("asm", lines of a statement) and ("code", instruction) in the order of the text."""
    label_at = {what: at for at, (kind, what) in enumerate(body) if kind == "label"}
    work = [at + 1 for at, (kind, what) in enumerate(body) if kind == "asm" and _after_statement(what)]
    seen, found = set(), set()
    while work:
        at = work.pop()
        while at < len(body) and at not in seen:
            seen.add(at)
            kind, what = body[at]
            at += 1
            if kind == "asm":
                if _after_statement(what) is not None:
                    break                         # it has waited, or its own reads start a path of their own
            elif kind == "code":
                if any(f == "v" and first < fragments_end for f, first, _ in _registers(what)):
                    found.add(at - 1)
                op = what.split()[0]
                if op in ("s_setpc_b64", "s_swappc_b64"):
                    raise RuntimeError(f"cannot follow {what}")
                if op == "s_endpgm":
                    break
                if op == "s_branch" or op.startswith("s_cbranch"):
                    work.append(label_at[what.split()[1]])
                    if op == "s_branch":
                        break
    return [body[at][1] for at in sorted(found)]


def check(asm_path: str) -> int:
    """Returns the number of checked kernels; raises on a collision."""
    kernel = None
    statement = None          # lines of the inline assembly being read
    checked = {}
    problems = []
    with open(asm_path) as f:
        for line in f:
            m = _KERNEL.match(line)
            if m:
                kernel = m.group(1)
                checked[kernel] = []
                continue
            if line.startswith("_Z") and _ANY_FN.match(line):
                kernel = None
                continue
            if kernel is None:
                continue
            body = checked[kernel]
            if ";;#ASMSTART" in line:
                statement = []
                continue
            if ";;#ASMEND" in line:
                body.append(("asm", statement))
                statement = None
                continue
            code = line.split(";")[0].strip()
            if statement is not None:
                statement.append(code)
                continue
            m = _LABEL.match(code)
            if m:
                body.append(("label", m.group(1)))
                continue
            if not code or code.startswith("."):
                continue
            body.append(("code", code))
            first_acc, first_vec = _owned_from(kernel)
            if any(last >= (first_acc if file_ == "a" else first_vec) for file_, _, last in _registers(code)):
                problems.append(f"{kernel}: {code}")
    if problems:
        raise RuntimeError(
            "the compiler placed values of its own in registers that belong to the kernel's assembly "
            f"({len(problems)} instructions), e.g.\n  " + "\n  ".join(problems[:8]))
    for kernel, body in checked.items():
        if _fragments_end(kernel):
            problems += [f"{kernel}: {code}" for code in _early_touches(body, _fragments_end(kernel))]
    if problems:
        raise RuntimeError(
            "the compiler uses registers of fragments whose LDS reads may still be in flight "
            f"({len(problems)} instructions), e.g.\n  " + "\n  ".join(problems[:8]))
    if not checked:
        raise RuntimeError(f"{asm_path}: no checked kernel found")
    return len(checked)


if __name__ == "__main__":
    for path in sys.argv[1:]:
        print(f"{path}: {check(path)} kernels, the assembly's registers untouched by the compiler")
