"""The global -> LDS DMA takes its LDS address from m0 and must not be issued in the instruction right after m0 is
written (no hardware interlock for the pair; inside inline assembly the compiler inserts nothing).  Every inline-assembly
string of the HIP sources that writes m0 and starts a DMA has a wait state between the two."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llmxabe_amd", "csrc")


def _dma_statements():
    for name in sorted(os.listdir(CSRC)):
        if not name.endswith((".hip", ".h")):
            continue
        text = open(os.path.join(CSRC, name)).read()
        for m in re.finditer(r'asm volatile\(\s*((?:"[^"]*"\s*)+)', text):
            lines = "".join(re.findall(r'"([^"]*)"', m.group(1))).replace("\\t", " ").split("\\n")
            ops = [l.split()[0] for l in lines if l.strip()]
            yield name, [l.strip() for l in lines], ops


def test_a_wait_state_separates_the_address_from_the_dma():
    seen = 0
    for name, lines, ops in _dma_statements():
        dma = [i for i, op in enumerate(ops) if "_load_lds_" in op]
        for i in dma:
            seen += 1
            wrote = [j for j in range(i) if re.match(r"s_mov_b32 m0\b", lines[j])]
            assert wrote, (name, "the DMA's address is set in the same statement", lines)
            assert i - wrote[-1] > 1, (name, "m0 is written in the instruction before the DMA", lines)
    assert seen >= 1
