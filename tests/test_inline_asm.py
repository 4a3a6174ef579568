"""Inline assembly of the kernels' sources: what a statement changes is among its clobbers."""

import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "byox_vllm_amd", "csrc")


def test_statements_that_write_m0_say_so():
    """The compiler keeps values of its own in m0 and does not look into the text."""
    found = 0
    for path in glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(CSRC, "*.hip")):
        with open(path) as f:
            for statement in re.findall(r"\basm(?: volatile)?\((.*?)\);", f.read(), re.S):
                if re.search(r"s_mov_b32 m0\b", statement):
                    found += 1
                    assert re.search(r':[^:]*"m0"[^:]*$', statement), f"{path}: {statement}"
    assert found
