"""Direct-to-LDS loads written in assembly take their LDS address from M0; the
ISA asks for one wait state between M0's write and such a load, and within an
assembly block the compiler adds none."""

import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hayate-exp_amd",
                    "csrc")


def test_a_wait_state_follows_every_write_of_m0():
    blocks = []
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h*"))):
        with open(path) as f:
            # adjacent string literals are one
            text = re.sub(r'"\s*"', "", f.read())
        blocks += [(path, b) for b in re.findall(r'__asm__ volatile\(\s*"([^"]*\bm0\b[^"]*)"', text)]
    assert len(blocks) >= 2
    for path, block in blocks:
        lines = [line.strip() for line in block.replace("\\t", " ").split("\\n")]
        writes = [i for i, line in enumerate(lines) if re.match(r"s_mov_b32 m0,", line)]
        assert writes, (path, block)
        for i in writes:
            assert lines[i + 1].startswith("s_nop"), (path, block)
