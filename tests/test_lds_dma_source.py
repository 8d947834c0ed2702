"""LDS-DMA is issued from inline asm, where hipcc adds no wait states: a write of m0 needs one before the load that reads it."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ipex_llm_amd", "csrc")


def test_m0_is_settled_before_the_load():
    found = 0
    for p in sorted(glob.glob(os.path.join(CSRC, "**", "*"), recursive=True)):
        if not p.endswith((".hip", ".cuh", ".h")):
            continue
        for asm in re.findall(r'asm volatile\(\s*"([^:]*?)"\s*:', open(p).read()):
            ops = [i.split()[0] for i in asm.replace("\\t", "").split("\\n") if i.strip()]
            for at, i in enumerate(ops):
                if "m0," in asm and i.startswith("buffer_load"):
                    found += 1
                    assert at >= 2 and ops[at - 1] == "s_nop", (p, asm)
    assert found
