"""Instructions that the compiler cannot see into (no GPU)."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "pytorch-transformers_amd", "csrc")


def test_no_arithmetic_in_inline_asm():
    """A matrix instruction's result may be read only some cycles after it was issued, and the compiler places the waits before the instructions that
    it knows: one in inline asm that reads scores or sums would read what the registers held before.  Loads, waits and moves of scalars stay."""
    bad = []
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(CSRC, "*.hip"))):
        with open(path) as f:
            text = f.read()
        for m in re.finditer(r'\basm\b(?:\s+volatile)?\s*\(\s*"([^"]*)"', text):
            if re.search(r"\bv_\w+", m.group(1)):
                bad.append(f"{os.path.basename(path)}: {m.group(1)}")
    assert not bad, bad
