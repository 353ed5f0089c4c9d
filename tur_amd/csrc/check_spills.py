#!/usr/bin/env python3
"""Build-time check that no kernel of a translation unit spills registers.

A kernel that runs out of registers still gives right results, from scratch memory, at a fraction of its speed, and nothing
says so: the build fails instead.  One that runs out of scalar registers keeps them in lanes of vector registers, a lane write and a
read for each, which shows neither.  hipcc prints the resources of every kernel with -Rpass-analysis=kernel-resource-usage; this
script reads those remarks and fails when a kernel uses scratch memory ("ScratchSize [bytes/lane]" above zero) or spills scalar
registers ("SGPRs Spill" above zero), unless its name matches one of the patterns below, which name the kernels that keep a small
array in private memory on purpose and those whose scalar spills are known.

usage: check_spills.py <file with the remarks> [<more files>]
"""
import re
import subprocess
import sys

# (what the remarks call it, pattern of the demangled name, the most that is accepted, why)
ALLOWED = [
    ("ScratchSize [bytes/lane]", r"\bdequant_tiled_kernel<", 256, "load time only: one thread rebuilds one native block in a private array, written for clarity"),
    ("ScratchSize [bytes/lane]", r"\bgather_tiled_kernel<", 256, "the same private block, for embedding rows of a table kept in the tiled layout"),
    ("SGPRs Spill", r"\bgemv_(mfma|multi_frag|gateup_frag|multi_frag_mixed)_kernel<", 250,
     "prepared fragments with several row tiles or column tiles in flight: the addresses of two m-tiles' fragments; accepted as it is"),
    ("SGPRs Spill", r"\bgemv_cs_staged_kernel<\d+, \d+, \d+, 32, 2, 0, false, (true|false)>", 8,
     "row addresses that a pair of column tiles shares: worked out for every column tile instead, the launches take 1 - 2 % longer (load_x_rows)"),
]
UNITS = {"ScratchSize [bytes/lane]": "bytes of scratch per lane", "SGPRs Spill": "scalar registers that are kept elsewhere"}


def demangle(names):
    if not names:
        return {}
    out = subprocess.run(["c++filt"], input="\n".join(names), capture_output=True, text=True, check=True).stdout.splitlines()
    return dict(zip(names, out))


def main(paths):
    found = []          # (file, mangled name, what, how much)
    kernels = 0
    for path in paths:
        name = None
        with open(path, errors="replace") as f:
            for line in f:
                m = re.search(r"Function Name: (\S+)", line)
                if m:
                    name = m.group(1)
                    kernels += 1
                    continue
                m = re.search(r"(ScratchSize \[bytes/lane\]|SGPRs Spill): (\d+)", line)
                if m and name and int(m.group(2)) > 0:
                    found.append((path, name, m.group(1), int(m.group(2))))
    readable = demangle(sorted({n for _, n, _, _ in found}))
    bad = []
    for path, name, what, much in found:
        text = readable.get(name, name)
        if not any(what == w and re.search(pat, text) and much <= most for w, pat, most, _ in ALLOWED):
            bad.append(f"{path}: {text[:160]} uses {much} {UNITS[what]}")
    if bad:
        print("check_spills: kernels that spill registers (or use private memory):", file=sys.stderr)
        for b in bad:
            print("  " + b, file=sys.stderr)
        return 1
    print(f"check_spills: {kernels} kernels in {len(paths)} file(s), none spills ({len(found)} as listed)")
    return 0


if __name__ == "__main__":
    if len(sys.argv) < 2:
        print(__doc__, file=sys.stderr)
        sys.exit(2)
    sys.exit(main(sys.argv[1:]))
