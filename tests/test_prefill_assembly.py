"""CPU: what the compiler cannot know about hand-written instructions of csrc/prefill.hip."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tidaldecode_amd", "csrc")


def test_m0_is_named_as_overwritten():
    with open(os.path.join(CSRC, "prefill.hip")) as f:
        statements = re.findall(r"asm volatile\((.*?)\);", f.read(), re.S)
    writes = [s for s in statements if "s_mov_b32 m0" in s]
    assert len(writes) == 2 and all('"m0"' in s.split(":")[-1] for s in writes)
