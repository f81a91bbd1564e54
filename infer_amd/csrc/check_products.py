"""Looks over the assembly of kernels that write matrix products as inline assembly.

    check_products.py FILE.s KERNEL

The compiler keeps the distances that matrix instructions need only between those that it knows, which are the products outside of inline assembly (where a
kernel has none marked, every product counts as written there).  For every instance of KERNEL in FILE.s
this reports, over all ways through the branches: a register copy or other vector instruction that writes an operand of a product less than
VALU_WAITS wait states in front of it; anything but the product itself that touches a product's result less than RESULT_WAITS behind it
(eight passes need 11, sixteen 19); and the use of scratch memory, where spilled accumulators would go.  Exit code 1 if there is any of it,
or no such kernel."""
import re
import sys

VALU_WAITS, RESULT_WAITS = 3, 19


def registers(operand):
    m = re.match(r"^([va])\[(\d+):(\d+)\]$", operand)
    if m:
        return {(m[1], i) for i in range(int(m[2]), int(m[3]) + 1)}
    m = re.match(r"^([va])(\d+)$", operand)
    return {(m[1], int(m[2]))} if m else set()


def operands(instruction):
    parts = instruction.split(None, 1)
    return [registers(o.strip().split(" ")[0]) for o in parts[1].split(",")] if len(parts) > 1 else []


def kernels(assembly, name):
    """(symbol, lines) of every instance."""
    lines = assembly.split("\n")
    for start, line in enumerate(lines):
        m = re.match(r"^(_Z\w*" + name + r"\w*|" + name + r"):", line)
        if m:
            end = next((j for j in range(start, len(lines)) if lines[j].startswith(".Lfunc_end")), len(lines))
            yield m[1], lines[start:end]


def parse(lines):
    """Instructions, for each the ones that may come in front of it, and the places of those in inline assembly."""
    code, labels, inline, inside = [], {}, set(), False
    for line in lines:
        if "#ASMSTART" in line or "#ASMEND" in line:
            inside = "#ASMSTART" in line
        line = line.split(";")[0].strip()
        m = re.match(r"^(\.L\w+):", line)
        if m:
            labels[m[1]] = len(code)
        elif line and not line.startswith(".") and not line.endswith(":"):
            if inside:
                inline.add(len(code))
            code.append(line)
    before = [[i - 1] if i and not code[i - 1].startswith(("s_branch", "s_endpgm", "s_setpc")) else [] for i in range(len(code))]
    for i, line in enumerate(code):
        m = re.match(r"s_c?branch\w*\s+(\.L\w+)", line)
        if m and labels.get(m[1], len(code)) < len(code):
            before[labels[m[1]]].append(i)
    return code, before, inline


def within(code, before, at, waits):
    """Instructions that may be issued fewer than `waits` wait states in front of `at`."""
    found, stack = set(), [(at, waits)]
    best = {}
    while stack:
        i, left = stack.pop()
        for p in before[i]:
            if left <= 0 or best.get(p, -1) >= left:
                continue
            best[p] = left
            found.add(p)
            m = re.match(r"s_nop (\d+)", code[p])
            stack.append((p, left - (int(m[1]) + 1 if m else 1)))
    return found


def product(line):
    return line.startswith(("v_mfma", "v_smfmac"))


def faults(lines):
    code, before, inline = parse(lines)
    found, products = [], {i for i, line in enumerate(code) if product(line)}
    written = products & inline or products                      # those between which the compiler keeps no distance
    for i, line in enumerate(code):
        used = operands(line)
        if i in written:
            read = set().union(*used[1:])
            for p in within(code, before, i, VALU_WAITS):
                if code[p].startswith("v_") and not product(code[p]) and operands(code[p]) and operands(code[p])[0] & read:
                    found.append(f"written right in front of a product: {code[p]} | {line}")
        touched = set().union(*used) if used else set()
        if touched and not line.startswith("s_"):
            for p in within(code, before, i, RESULT_WAITS):
                if p in products and (p in written or i in written) and operands(code[p])[0] & touched:
                    found.append(f"touches a product's result too early: {code[p]} | {line}")
    return found, len(written)


def scratch(assembly, symbol):
    """Bytes of scratch memory in the kernel's metadata; None: not stated."""
    m = re.search(r"\.amdhsa_kernel " + re.escape(symbol) + r"\n.*?\.amdhsa_private_segment_fixed_size (\d+)", assembly, re.S)
    return int(m[1]) if m else None


def check(assembly, name):
    found, seen = [], 0
    for symbol, lines in kernels(assembly, name):
        bad, products = faults(lines)
        seen += products > 0
        if scratch(assembly, symbol) != 0:
            bad.append(f"scratch memory: {scratch(assembly, symbol)} bytes")
        found += [f"{symbol}: {b}" for b in bad]
    return found if seen else found + [f"no kernel {name} with products"]


if __name__ == "__main__":
    with open(sys.argv[1]) as f:
        problems = check(f.read(), sys.argv[2])
    print("\n".join(problems[:20]))
    sys.exit(bool(problems))
