"""Dynamic local memory starts where the kernel's own variables end, at the alignment of its declared
type.  Declared as bytes it may start at any address, and FP64 accesses that straddle their eight bytes
cost several (the n = 320 FP64 inverse took 1386 us a level instead of 500)."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "chidg_amd", "csrc")


def test_byte_declarations_state_their_alignment():
    seen = 0
    for f in sorted(os.listdir(CSRC)):
        if not f.endswith(".hip"):
            continue
        for line in open(os.path.join(CSRC, f)):
            if re.search(r"extern __shared__.*\bchar\b", line):
                seen += 1
                assert re.search(r"aligned\(16\)|__align__\(16\)", line), f"{f}: {line.strip()}"
    assert seen
