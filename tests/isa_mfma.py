"""Check of the generated gfx950 code for the wait states of matrix instructions written in inline asm.

The compiler keeps the wait states between a matrix instruction and its neighbours only where it knows the instruction: one in an asm
statement is opaque to it, so whatever it places there by itself (an accumulator's zeros, a copy at a join of control flow, a register that
is used again) comes without them, and results are then wrong without an error.  Two rules, followed over every path of a kernel:
  * a vector instruction that writes a register stands at least two wait states in front of an asm matrix instruction that reads it;
  * for as many wait states as its result takes, nobody but a matrix instruction that adds to the same accumulator names a destination
    register of an asm matrix instruction.
An instruction is one wait state, `s_nop n` is n + 1 (waits for memory and barriers last longer than that and count as one).
"""
import re

# wait states between a matrix instruction of four passes and a reader or writer of its result, and behind a vector write, as the compiler keeps
# them for its own
RESULT = {"v_mfma_i32_16x16x64_i8": 8, "v_mfma_f32_16x16x32_f16": 8}
OPERAND = 2


def _regs(tok):
    out = set()
    for m in re.finditer(r"\b([va])\[(\d+):(\d+)\]|\b([va])(\d+)\b", tok):
        if m.group(1):
            out |= {m.group(1) + str(i) for i in range(int(m.group(2)), int(m.group(3)) + 1)}
        else:
            out.add(m.group(4) + m.group(5))
    return out


def _blocks(lines, first, last):
    """[(instructions, indices of the blocks that may follow)]; an instruction is (line number, text, stands in asm)."""
    blocks, names, cur, in_asm = [], {}, [], False
    ends = []  # per block: (label of a branch or None, falls through)
    for i in range(first, last):
        text = lines[i].split(";")[0].strip() if not lines[i].strip().startswith(";;#") else lines[i].strip()
        if text.startswith(";;#ASMSTART"):
            in_asm = True
        elif text.startswith(";;#ASMEND"):
            in_asm = False
        elif re.match(r"^\.?\w+:$", text) and not text.startswith("_Z"):
            blocks.append(cur)
            ends.append((None, True))
            names[text[:-1]] = len(blocks)
            cur = []
        elif text and not text.startswith((".", "_Z")):
            cur.append((i + 1, text, in_asm))
            op = text.split()[0]
            if op.startswith(("s_branch", "s_cbranch")) or op == "s_endpgm":
                blocks.append(cur)
                ends.append((text.split()[1] if op != "s_endpgm" else None, op.startswith("s_cbranch")))
                cur = []
    blocks.append(cur)
    ends.append((None, False))
    out = []
    for n, (label, falls) in enumerate(ends):
        after = [names[label]] if label in names else []
        if falls and n + 1 < len(blocks):
            after.append(n + 1)
        out.append((blocks[n], after))
    return out


def _step(state, block, found):
    """state: ({register: (wait states to go, line)} of asm matrix results, the same of vector writes), at the end of the block."""
    result, written = dict(state[0]), dict(state[1])
    for line, text, in_asm in block:
        op, _, rest = text.partition(" ")
        operands = [_regs(o) for o in rest.split(",")]
        named = set().union(*operands) if operands else set()
        matrix = op.startswith(("v_mfma", "v_smfmac"))
        own = in_asm and matrix
        if own and op not in RESULT:
            found.add((line, text, "how long its result takes is not known", 0))
        sums = operands[0] if own and operands[0] == operands[3] else set()
        for reg in named - sums:
            if reg in result:
                found.add((line, text, "names the result of a matrix instruction too early", result[reg][1]))
        for reg in sums:  # the same accumulator as a whole, or none of it
            if reg in result and result[reg][2] != sums:
                found.add((line, text, "adds to a part of a result in flight", result[reg][1]))
        if own:
            for reg in named:
                if reg in written:
                    found.add((line, text, "reads what was written just before", written[reg][1]))
        states = int(rest.split()[0], 0) + 1 if op == "s_nop" else 1
        result = {r: (v[0] - states,) + v[1:] for r, v in result.items() if v[0] > states}
        written = {r: (v[0] - states,) + v[1:] for r, v in written.items() if v[0] > states}
        if own:
            for reg in operands[0]:
                result[reg] = (RESULT.get(op, 0), line, frozenset(operands[0]))
        elif op.startswith("v_") and not matrix:
            for reg in operands[0] | (operands[1] if "swap" in op and len(operands) > 1 else set()):
                written[reg] = (OPERAND, line)
    return result, written


def _join(a, b):
    out = []
    for x, y in zip(a, b):
        both = dict(x)
        for reg, v in y.items():
            if reg not in both or both[reg][0] < v[0]:
                both[reg] = v
        out.append(both)
    return tuple(out)


def broken_wait_states(asm_text):
    """[(kernel, line, instruction, what is wrong, line of the other instruction)]"""
    lines = asm_text.split("\n")
    starts = [(i, l.split(":")[0]) for i, l in enumerate(lines) if re.match(r"^_Z\w+:", l)]
    report = []
    for n, (first, name) in enumerate(starts):
        blocks = _blocks(lines, first, starts[n + 1][0] if n + 1 < len(starts) else len(lines))
        entry = {0: ({}, {})}
        work, found = [0], set()
        while work:
            b = work.pop()
            end = _step(entry[b], blocks[b][0], found)
            for after in blocks[b][1]:
                state = _join(entry[after], end) if after in entry else end
                if state != entry.get(after):
                    entry[after] = state
                    work.append(after)
        report += [(name,) + f for f in sorted(found)]
    return report


def asm_matrix_instructions(asm_text):
    """{mnemonic: count} of the matrix instructions in asm statements."""
    out, in_asm = {}, False
    for l in asm_text.split("\n"):
        l = l.strip()
        if l.startswith(";;#ASMSTART"):
            in_asm = True
        elif l.startswith(";;#ASMEND"):
            in_asm = False
        elif in_asm and l.startswith(("v_mfma", "v_smfmac")):
            out[l.split()[0]] = out.get(l.split()[0], 0) + 1
    return out
