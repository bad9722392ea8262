"""Reads the AMD assembly of sources that use acc_tiles.h and fails where a kernel's sums are not safe in their named registers.

The compiler does not know what the assembly on a[..] does: between two statements it takes those registers for free, and its hazard
pass does not look inside.  So in every kernel with an assembly MFMA on a named accumulator:
  * no instruction of the compiler's own names an accumulation register (a copy, a spill, a load into one);
  * nothing is spilled to memory and no function is called;
  * no vector instruction writes an operand of such an MFMA less than two wait states ahead of it (the compiler's own copies; LDS reads are waited for).
Usage: check_acc.py FILE.s ...; every file has to hold at least one such kernel."""
import re
import sys

ACC = re.compile(r"(?<![\w.$])a(\d+\b|\[\d+(:\d+)?\])")
VGPR = re.compile(r"^v(?:(\d+)|\[(\d+):(\d+)\])$")


def vector_registers(operand):
    m = VGPR.match(operand)
    if not m:
        return set()
    return {int(m[1])} if m[1] else set(range(int(m[2]), int(m[3]) + 1))


def functions(text):
    """(name, [(line number, instruction, written as assembly)], {directive: value}) of each function and its kernel descriptor."""
    found, name, in_asm, described = {}, None, False, None
    for number, line in enumerate(text.splitlines(), 1):
        if "ASMSTART" in line or "ASMEND" in line:
            in_asm = "ASMSTART" in line
            continue
        code = line.split(";")[0].strip()
        label = re.match(r"^([\w$.]+):", line)
        if label and not label[1].startswith("."):
            name = label[1]
            found.setdefault(name, ([], {}))
        elif code.startswith(".amdhsa_kernel"):
            described = code.split()[1]
            found.setdefault(described, ([], {}))
        elif code.startswith(".end_amdhsa_kernel"):
            described = None
        elif described and code.startswith(".amdhsa_"):
            key, value = code.split()[:2]
            found[described][1][key] = value
        elif name and re.match(r"^[a-z]\w*(\s|$)", code):
            found[name][0].append((number, code, in_asm))
    return [(n, code, info) for n, (code, info) in found.items()]


def faults(text):
    """Faults of the kernels that keep sums in named accumulators, and how many such kernels there are."""
    out, kernels = [], 0
    for name, code, info in functions(text):
        if not any(asm and c.startswith("v_mfma") and ACC.search(c.split(None, 1)[1].split(",")[0]) for _, c, asm in code):
            continue
        kernels += 1
        if info.get(".amdhsa_private_segment_fixed_size", "0") != "0":
            out.append(f"{name}: {info['.amdhsa_private_segment_fixed_size']} bytes of scratch")
        for i, (number, c, asm) in enumerate(code):
            op, operands = (c.split(None, 1) + [""])[:2]
            if op.startswith(("s_swappc", "s_call", "scratch_")):
                out.append(f"{name}, line {number}: {c}")
            if not asm and ACC.search(operands):
                out.append(f"{name}, line {number}: the compiler's own use of an accumulation register: {c}")
            if asm and op.startswith("v_mfma"):
                reads = set().union(*(vector_registers(o.strip()) for o in operands.split(",")[1:3]))
                states = 0
                for before, b, _ in reversed(code[max(0, i - 2):i]):
                    if states >= 2:
                        break
                    bop, boperands = (b.split(None, 1) + [""])[:2]
                    if bop.startswith("v_") and not bop.startswith(("v_mfma", "v_cmp")) and vector_registers(boperands.split(",")[0].strip()) & reads:
                        out.append(f"{name}, line {before}: {b}, {states} wait states ahead of {c}")
                    states += int(boperands, 0) + 1 if bop == "s_nop" else 1
    return out, kernels


def main(paths):
    bad = 0
    for path in paths:
        with open(path) as f:
            found, kernels = faults(f.read())
        if not kernels:
            found.append("no kernel with sums in named accumulators found")
        for fault in found:
            print(f"{path}: {fault}", file=sys.stderr)
        bad += len(found)
    return bad != 0


if __name__ == "__main__":
    sys.exit(main(sys.argv[1:]))
