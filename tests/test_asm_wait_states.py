"""CPU: the wait states that hand-written instructions have to bring along, in the assembly of csrc/topk.hip and
csrc/gemm.hip (compiled here, about 15 seconds: without optimisation, which the text of a statement does not
depend on).

Inside an asm statement the compiler inserts none.  gfx950 needs two between a vector instruction that writes a
scalar pair (a comparison's mask) and a vector instruction that reads it as a mask or carry, one between the
write of m0 and a load to LDS, and five between a vector instruction that writes a scalar register and the load
that takes it as its base."""
import os
import re
import subprocess

import pytest

from test_prefill_assembly import CSRC, HIPCC, _wait_states


@pytest.fixture(scope="module")
def blocks(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    out = {}
    for name in ("topk", "gemm"):
        path = str(tmp_path_factory.mktemp("asm") / f"{name}.s")
        subprocess.run([HIPCC, "--offload-arch=gfx950", "-O0", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "--cuda-device-only", "-S", os.path.join(CSRC, f"{name}.hip"), "-o", path],
                       check=True, stderr=subprocess.DEVNULL)
        with open(path) as f:
            found = re.findall(r";;#ASMSTART\n(.*?);;#ASMEND", f.read(), re.S)
        out[name] = [[i.strip() for i in b.split("\n") if i.strip()] for b in found]
    return out


def _masks(instruction):
    """the scalar pairs that a vector instruction writes and reads"""
    op, _, rest = instruction.partition(" ")
    args = [a.strip() for a in re.split(r",(?![^\[]*\])", rest)]
    if not op.startswith("v_"):
        return set(), set()
    scalar = lambda xs: {x for x in xs if x == "vcc" or x.startswith("s[")}
    if op.startswith("v_cmp"):
        return scalar(args[:1]), scalar(args[1:])
    return scalar(args[:2]), scalar(args[2:])


def short_waits(block):
    """the instructions of an asm block that read a mask less than two wait states after it was written"""
    bad = []
    for n, i in enumerate(block):
        for back in range(n - 1, -1, -1):
            if _wait_states(block[back + 1 : n]) >= 2:
                break
            if _masks(block[back])[0] & _masks(i)[1]:
                bad.append((block[back], i))
    return bad


def test_the_check_itself():
    compare, add = "v_cmp_nlt_f32 vcc, v1, v2", "v_addc_co_u32 v0, vcc, v0, v0, vcc"
    assert short_waits([compare, add]) and short_waits([compare, "s_nop 0", add])
    assert not short_waits([compare, "s_nop 1", add])
    assert short_waits(["v_cmp_nlt_f32 s[4:5], v1, v2", "v_cmp_nlt_f32 s[6:7], v1, v2",
                        "v_addc_co_u32 v0, s[4:5], v0, v0, s[4:5]"])


def test_masks_are_read_two_wait_states_after_they_are_written(blocks):
    compares = [b for b in blocks["topk"] if any(i.startswith("v_cmp") for i in b)]
    assert len(compares) >= 3 * 3  # three types, the three kernels whose rows may be longer than the sample
    for b in compares:
        assert not short_waits(b), b


def test_loads_to_lds_bring_their_wait_states_along(blocks):
    loads = [b for b in blocks["gemm"] if b and "global_load_lds" in b[-1]]
    assert len(loads) >= 2  # two types
    for b in loads:
        at = next(n for n, i in enumerate(b) if i.startswith("s_mov_b32 m0"))
        assert _wait_states(b[at + 1 : -1]) >= 1 and _wait_states(b[:-1]) >= 5, b


def test_m0_is_named_as_overwritten():
    with open(os.path.join(CSRC, "gemm.hip")) as f:
        statements = re.findall(r"asm volatile\((.*?)\);", f.read(), re.S)
    writes = [s for s in statements if "s_mov_b32 m0" in s]
    assert len(writes) == 1 and '"m0"' in writes[0].split(":")[-1]
