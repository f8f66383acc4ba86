"""Checks the assembly of the kernels that keep accumulators in AccVGPRs by hand (csrc/qfa_acc.h), as the compiler wrote it.

Their inline MFMAs name AccVGPRs that the compiler does not know to hold anything between two statements, and it does not
see these MFMAs' hazards.  So the build looks at what it made of them:

  1. no instruction of the compiler's touches a register that holds an accumulator of inline assembly, between the statements or
     anywhere else, and none reads one that inline assembly has overwritten (it may use the others, and in a part of the kernel that
     shares no path with these statements all);
  2. a vector instruction that writes A or B of an inline MFMA is followed by at least two wait states before it, and one that
     writes an accumulator likewise;
  3. an accumulator is read, or written by a vector instruction, no earlier than 20 wait states behind an MFMA that writes it;
  4. these kernels spill nothing: an LDS request that the compiler does not know of may not have its registers moved.

    python -m quant_flash_attn_amd.acc_check FILE.s
"""
from __future__ import annotations

import re
import sys
from typing import Dict, List, NamedTuple, Set, Tuple

VALU_TO_MFMA = 2     # wait states between a vector instruction and an MFMA that reads what it wrote
MFMA_TO_VALU = 20    # ... between a 32x32 MFMA (16 passes) and a vector instruction on its result

_REG = re.compile(r"\b([va])(?:(\d+)\b|\[(\w+)(?::(\w+))?\])")


class Instr(NamedTuple):
    line: int
    text: str
    op: str
    inline: bool       # from an inline assembly statement
    writes: frozenset  # registers written, as ("v" | "a", number)
    reads: frozenset
    target: str        # label of a branch


def _regs(text: str) -> Set[Tuple[str, int]]:
    out = set()
    for m in _REG.finditer(text):
        if m.group(2) is not None:
            out.add((m.group(1), int(m.group(2))))
        else:
            out |= {(m.group(1), r) for r in range(int(m.group(3), 0), int(m.group(4) or m.group(3), 0) + 1)}
    return out


def _parse_instr(line: int, text: str, inline: bool) -> Instr:
    op, _, rest = text.partition(" ")
    ops = [x for x in re.split(r",\s*(?![^\[]*\])", rest.strip()) if x]
    stores = re.match(r"(ds_write|ds_store|global_store|buffer_store|scratch_store|flat_store|s_)", op) or "lds" in rest.split()
    dst = set() if stores or not ops else _regs(ops[0])
    src = set().union(*map(_regs, ops if stores else ops[1:])) if ops else set()
    if "swap" in op and len(ops) > 1:
        dst |= _regs(ops[1])
        src |= _regs(ops[0])
    if re.match(r"v_(dot2c|fmac|pk_fmac|mac)_", op):
        src |= dst
    return Instr(line, text, op, inline, frozenset(dst), frozenset(src), ops[0] if ops and op.startswith(("s_branch", "s_cbranch")) else "")


def _kernels(path: str):
    """(name, instructions, label -> index, bytes of scratch) of every kernel in an assembly file."""
    name, instrs, labels, inline = None, [], {}, False
    with open(path) as f:
        for n, raw in enumerate(f, 1):
            if "ASMSTART" in raw or "ASMEND" in raw:
                inline = "ASMSTART" in raw
                continue
            text = raw.split(";")[0].strip()
            m = re.match(r"([.\w$]+):$", text)
            if m:
                if m.group(1).startswith("_Z"):
                    name, instrs, labels = m.group(1), [], {}
                labels[m.group(1)] = len(instrs)
            elif name and text and not text.startswith("."):
                for part in text.split("\n"):
                    instrs.append(_parse_instr(n, part.strip().replace("\t", " "), inline))
            elif name and text.startswith(".amdhsa_private_segment_fixed_size"):
                yield name, instrs, labels, int(text.split()[1])
                name = None


def _wait_states(i: Instr) -> int:
    return int(i.text.split()[1], 0) + 1 if i.op == "s_nop" else 1


def check(path: str) -> List[str]:
    """What is wrong, one line each; empty: nothing."""
    bad: List[str] = []
    for name, ins, labels, scratch in _kernels(path):
        acc = {r for i in ins if i.inline for r in i.reads | i.writes if r[0] == "a"}
        if not acc:
            continue
        tell = lambda i, what: bad.append(f"{path}:{i.line}: {name}: {what}: {i.text}")   # noqa: E731
        if scratch:
            bad.append(f"{path}: {name}: {scratch} bytes of scratch")
        before: Dict[int, List[int]] = {}
        for k, i in enumerate(ins):
            if k + 1 < len(ins) and i.op not in ("s_branch", "s_endpgm", "s_setpc_b64"):
                before.setdefault(k + 1, []).append(k)
            if i.target in labels:
                before.setdefault(labels[i.target], []).append(k)

        # For each instruction, as bits: the accumulators that inline assembly may read from there on before it writes them anew, and those
        # that it has written since the compiler last did, on any path.  (A kernel may hold two loops of which a workgroup runs one:
        # registers of one are the compiler's in the other.)
        after: Dict[int, List[int]] = {}
        for k, ps in before.items():
            for p in ps:
                after.setdefault(p, []).append(k)
        bits = lambda regs: sum(1 << n for kind, n in regs if kind == "a")  # noqa: E731
        reads, writes = [bits(i.reads & acc) for i in ins], [bits(i.writes & acc) for i in ins]

        def flow(gen: List[int], kill: List[int], to: Dict[int, List[int]], order) -> List[int]:
            """What arrives at each instruction: gen and whatever arrived without kill goes on along the edges."""
            arrived, todo = [0] * len(ins), list(order)
            while todo:
                k = todo.pop()
                out = gen[k] | arrived[k] & ~kill[k]
                for n in to.get(k, []):
                    if out & ~arrived[n]:
                        arrived[n] |= out
                        todo.append(n)
            return arrived

        by_asm = lambda x: [b if i.inline else 0 for b, i in zip(x, ins)]   # noqa: E731
        wanted = flow(by_asm(reads), by_asm(writes), before, range(len(ins)))
        dirty = flow(by_asm(writes), [0 if i.inline else w for w, i in zip(writes, ins)], after, reversed(range(len(ins))))

        def written_within(k: int, regs, states: int, writer) -> bool:
            """Is there a path on which an instruction `writer` accepts writes one of `regs` fewer than `states` before k?"""
            todo, seen = [(p, states) for p in before.get(k, [])], {}
            while todo:
                p, left = todo.pop()
                if left <= 0 or seen.get(p, 0) >= left:
                    continue
                seen[p] = left
                if writer(ins[p]) and ins[p].writes & regs:
                    return True
                todo += [(q, left - _wait_states(ins[p])) for q in before.get(p, [])]
            return False

        mfma = lambda i: i.op.startswith("v_mfma")                          # noqa: E731
        valu = lambda i: i.op.startswith("v_") and not mfma(i)              # noqa: E731
        for k, i in enumerate(ins):
            used = i.reads | i.writes
            if not i.inline and ((reads[k] | writes[k]) & wanted[k] or reads[k] & dirty[k]):
                tell(i, "the compiler uses an accumulator's register")
            if i.inline and mfma(i):
                if written_within(k, i.reads | i.writes, VALU_TO_MFMA, valu):
                    tell(i, f"an operand is written less than {VALU_TO_MFMA} wait states earlier")
                if written_within(k, {r for r in i.reads if r[0] == "v"}, MFMA_TO_VALU, mfma):
                    tell(i, "an operand is the result of an MFMA that may not have finished")
            elif i.inline and valu(i) and written_within(k, used & acc, MFMA_TO_VALU, mfma):
                tell(i, f"an accumulator is used less than {MFMA_TO_VALU} wait states behind its MFMA")
    return bad


if __name__ == "__main__":
    found = [b for path in sys.argv[1:] for b in check(path)]
    print("\n".join(found) or "nothing found")
    sys.exit(1 if found else 0)
