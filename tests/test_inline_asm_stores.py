"""Stores of more than 64 bits written as inline assembly carry the two wait states in which their data must not be overwritten: the compiler
adds these only to stores that it knows."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "z-ant_amd", "csrc")


def test_wide_stores_in_inline_assembly_are_followed_by_their_wait_states():
    wide = []
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h*"))):
        with open(path) as f:
            for asm in re.findall(r'asm(?:\s+volatile)?\s*\(\s*((?:"(?:[^"\\]|\\.)*"\s*)+)', f.read()):
                for m in re.finditer(r"(?:global|buffer|flat|scratch)_store_\w*(?:x3|x4|96|128)\b", asm):
                    wide.append((os.path.basename(path), asm))
                    after = asm[m.end():].split("\\n", 1)
                    assert len(after) == 2 and re.match(r"(?:\\t|\s)*s_nop [1-9]", after[1]), (path, asm)
    assert {name for name, _ in wide} >= {"common.h", "conv_f32.hip"}, wide
