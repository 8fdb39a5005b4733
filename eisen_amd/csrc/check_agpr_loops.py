"""Checks the assembly of a HIP source for what its inline-assembly MFMAs rely on (attention_bwd.hip, mfma_agpr).

The compiler does not see an MFMA in inline assembly and so does not wait for its result.  That is sound as long as, in the
loop around such MFMAs, nothing else touches their accumulators (AGPRs) and nothing is spilled, and behind the loop nothing
reads them before the wait states of agpr_settle().  Register allocation decides both, so the build looks:

    python3 check_agpr_loops.py attention_bwd.s kernel-name-part number-of-kernels
"""
import re
import sys

MFMA = re.compile(r"\bv_mfma\w*\s+a\[")
AGPR = re.compile(r"accvgpr|\ba\[\d|\ba\d+\b")
SPILL = re.compile(r"\bscratch_(load|store)")
BRANCH = re.compile(r"\b(s_c?branch\w*)\s+(\.LBB\w+)")
SETTLE = re.compile(r"\bs_nop\s+(15|0xf)\b")


def functions(text):
    """(name, lines) of every function of an assembly listing, comments left out."""
    for m in re.finditer(r"^(\w+):[^\n]*\n(.*?)^\.Lfunc_end\d+:", text, re.S | re.M):
        yield m.group(1), [re.sub(r"(?<!;);(?!;).*", "", line) for line in m.group(2).split("\n")]


def asm_mfmas(lines):
    """Line numbers of the AGPR MFMAs that stand between the markers of inline assembly."""
    found, inside = [], False
    for i, line in enumerate(lines):
        if "ASMSTART" in line:
            inside = True
        elif "ASMEND" in line:
            inside = False
        elif inside and MFMA.search(line):
            found.append(i)
    return found


def problems(lines):
    mfmas = asm_mfmas(lines)
    labels = {m.group(1): i for i, line in enumerate(lines) if (m := re.match(r"(\.LBB\w+):", line))}
    loops = []  # backward branches around all of them
    for i, line in enumerate(lines):
        m = BRANCH.search(line)
        if m and i > mfmas[-1] and labels.get(m.group(2), i) <= mfmas[0]:
            loops.append((i - labels[m.group(2)], labels[m.group(2)], i))
    if not loops:
        return ["no loop around the MFMAs"]
    _, first, last = min(loops)
    out = []
    for i in range(first, last + 1):
        if SPILL.search(lines[i]):
            out.append(f"scratch access in the loop: {lines[i].strip()}")
        if AGPR.search(lines[i]) and i not in mfmas:
            out.append(f"accumulator register in use in the loop: {lines[i].strip()}")
    # every way out of the loop: branches to a label outside of it, and falling out of its end
    exits = {last + 1} if "s_cbranch" in lines[last] else set()
    for line in lines[first:last + 1]:
        m = BRANCH.search(line)
        if m and not first <= labels.get(m.group(2), first) <= last:
            exits.add(labels[m.group(2)])
    for i in sorted(exits):
        for _ in range(len(lines)):
            if i >= len(lines):
                out.append("no wait states behind the loop")
                break
            if SETTLE.search(lines[i]):
                break
            if AGPR.search(lines[i]):
                out.append(f"accumulator register in use behind the loop before the wait states: {lines[i].strip()}")
                break
            m = BRANCH.search(lines[i])
            i = labels.get(m.group(2), len(lines)) if m and m.group(1) == "s_branch" else i + 1
    return out


def check(text, name_part, expected):
    """Messages, empty if all is well."""
    kernels = [(name, lines) for name, lines in functions(text) if name_part in name and asm_mfmas(lines)]
    out = [] if len(kernels) == expected else [f"{len(kernels)} kernels {name_part} with inline-assembly MFMAs, expected {expected}"]
    for name, lines in kernels:
        out += [f"{name}: {p}" for p in problems(lines)]
    return out


if __name__ == "__main__":
    bad = check(open(sys.argv[1]).read(), sys.argv[2], int(sys.argv[3]))
    print("\n".join(bad), file=sys.stderr) if bad else None
    sys.exit(1 if bad else 0)
