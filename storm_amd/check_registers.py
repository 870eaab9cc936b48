"""Checks the compiler's resource remarks for the transport kernels.

    check_registers.py REMARKS

REMARKS is what hipcc prints with -Rpass-analysis=kernel-resource-usage.
Exits 1, naming the kernels, if a transport kernel spills vector registers or
uses scratch memory, or if the remarks hold none.  A build of an earlier form
of these kernels that spilled 100 bytes counted escapes and walk steps wrongly
(kernels.h, TransportWaves).
"""
import re
import sys


def kernels(text):
    """{mangled name: {resource: number}} of every function with remarks."""
    out, cur = {}, None
    for line in text.splitlines():
        m = re.search(r"remark: (.*?)(?: \[-Rpass-analysis=kernel-resource-usage\])?$", line)
        if not m:
            continue
        key, _, value = m.group(1).rpartition(":")
        key, value = key.strip().split(": ")[-1], value.strip()
        if key.endswith("Function Name"):
            cur = out.setdefault(value, {})
        elif cur is not None and value.isdigit():
            cur[key] = int(value)
    return out


def problems(text):
    found = {k: v for k, v in kernels(text).items() if "k_transport" in k}
    if not found:
        return ["no transport kernel in the remarks"]
    bad = []
    for name, r in found.items():
        spill, scratch = r.get("VGPRs Spill"), r.get("ScratchSize [bytes/lane]")
        if spill != 0 or scratch != 0:
            bad.append(f"{name}: {spill} vector registers spilled, {scratch} bytes of scratch a lane")
    return bad


if __name__ == "__main__":
    with open(sys.argv[1]) as f:
        bad = problems(f.read())
    for line in bad:
        print(line, file=sys.stderr)
    sys.exit(1 if bad else 0)
