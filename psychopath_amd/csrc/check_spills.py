"""Fails on device assembly that spills a vector register where lanes are
missing.

    python3 check_spills.py FILE.s ...

Where two sides of a branch meet, the block gives the lanes their turn back
(`s_or_b64 exec` or `s_or_saveexec_b64`) before it does anything else.  The
compiler has placed register spills ahead of that: the lanes of the other side
then never store their value and later reload whatever the slot held.  A
shading build for three waves per SIMD lost the emission of light hits so (one
block of 18,470), and no change to the source states that it must not.
"""

import re
import sys

KERNEL = re.compile(r"^([A-Za-z_]\w*):[^\n]*\n(.*?)^\.Lfunc_end", re.S | re.M)
LABEL = re.compile(r"\.LBB\d+_\d+:")
SPILL = re.compile(r"scratch_store_\w+ off, .*Spill|v_accvgpr_write_b32")
# what may stand between the label and the spills of such a block
HEAD = re.compile(r"s_waitcnt|s_nop|s_mov_b|v_mov_b|v_readlane_b32|v_writelane_b32|scratch_load_\w+ .*Reload")
RESTORE = re.compile(r"s_or_b64 exec, exec,|s_or_saveexec_b64")


def early_spills(asm: str) -> list:
    """(kernel, label, spill) of every spill ahead of its block's restore."""
    found = []
    for kernel, body in KERNEL.findall(asm):
        label, spills = None, []
        for line in body.split("\n"):
            if LABEL.match(line):
                label, spills = line.split(":")[0], []
                continue
            s = line.strip()
            if label is None or not s or s.startswith(";"):
                continue
            if SPILL.match(s):
                spills.append(s.split(";")[0].strip())
            elif not HEAD.match(s):
                if RESTORE.match(s):
                    found += [(kernel, label, x) for x in spills]
                label = None
    return found


def main(paths: list) -> int:
    bad = 0
    for path in paths:
        with open(path) as f:
            for kernel, label, spill in early_spills(f.read()):
                print(f"{path}: {kernel} {label}: '{spill}' stands before the lanes' mask is restored",
                      file=sys.stderr)
                bad += 1
    return 1 if bad else 0


if __name__ == "__main__":
    raise SystemExit(main(sys.argv[1:]))
