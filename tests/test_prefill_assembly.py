"""CPU: hazards that the compiler leaves to hand-written instructions, and the registers of the kernels,
checked in the assembly of csrc/prefill.hip (compiled here, about four seconds).

Inside an asm statement the compiler inserts no wait states.  gfx950 needs five between a vector
instruction that writes a scalar register (v_readlane, v_readfirstlane) and a memory instruction that
reads it, and one between the write of m0 and a load to LDS."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tidaldecode_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    out = str(tmp_path_factory.mktemp("asm") / "prefill.s")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "--cuda-device-only", "-S", os.path.join(CSRC, "prefill.hip"), "-o", out],
                   check=True, stderr=subprocess.DEVNULL)
    with open(out) as f:
        return f.read()


@pytest.fixture(scope="module")
def asm_blocks(assembly):
    return [[i.strip() for i in b.split("\n") if i.strip()]
            for b in re.findall(r";;#ASMSTART\n(.*?);;#ASMEND", assembly, re.S)]


def _wait_states(instructions):
    return sum(int(i.split()[1]) + 1 if i.startswith("s_nop") else 1 for i in instructions)


def test_loads_to_lds_bring_their_wait_states_along(asm_blocks):
    loads = [b for b in asm_blocks if b and "global_load_lds" in b[-1]]
    assert len(loads) >= 100                      # four kernels of 64 and 128 dimensions, two types
    assert any("s[" in b[-1] for b in loads) and any(b[-1].endswith("off") for b in loads)
    for b in loads:
        at = next(n for n, i in enumerate(b) if i.startswith("s_mov_b32 m0"))
        assert _wait_states(b[at + 1 : -1]) >= 1, b
        if "s[" in b[-1]:                         # the base may come from v_readlane right before
            assert _wait_states(b[:-1]) >= 5, b


def test_m0_is_named_as_overwritten():
    with open(os.path.join(CSRC, "prefill.hip")) as f:
        statements = re.findall(r"asm volatile\((.*?)\);", f.read(), re.S)
    writes = [s for s in statements if "s_mov_b32 m0" in s]
    assert len(writes) == 2 and all('"m0"' in s.split(":")[-1] for s in writes)


def test_two_waves_of_an_attention_kernel_share_a_simd(assembly):
    """Eight waves of 64 / 128 dimensions and two workgroups of 256 dimensions per compute unit need kernels
    of at most 256 registers; more puts the accumulators into the second register file, with copies in
    every step."""
    kernels = re.findall(r"^(\S*prefill_attn\S*):[^\n]*\n(.*?)\.end_amdhsa_kernel", assembly, re.S | re.M)
    assert len(kernels) == 2 * (4 + 3)
    for name, body in kernels:
        assert int(re.search(r"\.amdhsa_next_free_vgpr (\d+)", body).group(1)) <= 256, name
        assert "scratch_" not in body and "v_accvgpr" not in body, name


def test_attention_kernels_divide_by_multiplication(assembly):
    """A division by a run-time number starts with v_rcp_iflag_f32 and is a chain of some 20 instructions."""
    for name, body in re.findall(r"^(\S*prefill_attn\S*):[^\n]*\n(.*?)\.end_amdhsa_kernel", assembly, re.S | re.M):
        assert "v_rcp_iflag" not in body, name
