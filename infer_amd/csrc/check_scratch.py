"""Looks over the compiler's report on the resources of kernels (-Rpass-analysis=kernel-resource-usage).

    check_scratch.py REPORT NAME=SPILLS ...

An instance of a kernel, by its mangled symbol, is held to the first NAME that is a part of it: no more than SPILLS of its vector registers may be spilled.
Exit code 1 if one has more, or a NAME meets no instance."""
import re
import sys


def instances(report):
    """Symbol -> spilled vector registers."""
    return {m[1]: int(m[2]) for m in re.finditer(r"Function Name: (\S+)(?:(?!Function Name:).)*?VGPRs Spill: (\d+)", report, re.S)}


def check(report, limits):
    found, met = [], set()
    for symbol, spills in instances(report).items():
        name = next((n for n in limits if n in symbol), None)
        if name is not None:
            met.add(name)
            if spills > limits[name]:
                found.append(f"{symbol}: {spills} vector registers spilled, {limits[name]} allowed")
    return found + [f"no kernel {n}" for n in limits if n not in met]


if __name__ == "__main__":
    with open(sys.argv[1]) as f:
        problems = check(f.read(), {n: int(k) for n, k in (a.split("=") for a in sys.argv[2:])})
    print("\n".join(problems[:20]))
    sys.exit(bool(problems))
