"""What the compiler made of the kernels, read from the built code object (llvm-objdump on this library's own gfx950 code)."""
import os
import re
import subprocess

import pytest

import gi_attn

LLVM = "/opt/rocm/llvm/bin"


@pytest.fixture(scope="module")
def code_object(tmp_path_factory):
    if not os.path.exists(f"{LLVM}/clang-offload-bundler"):
        pytest.skip("no LLVM tools")
    out = tmp_path_factory.mktemp("co") / "gi_attn.o"
    subprocess.run([f"{LLVM}/clang-offload-bundler", "--unbundle", "--type=o", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950",
                    f"--input={gi_attn.HSACO_PATH}", f"--output={out}"], check=True)
    return str(out)


def test_no_load_loops_over_the_lanes_descriptors(code_object):
    # a buffer descriptor that the compiler keeps in vector registers turns each load into a loop that masks the lanes
    # with equal descriptors (v_readfirstlane, v_cmp, s_and_saveexec, buffer_load, s_cbranch_execnz)
    asm = subprocess.run([f"{LLVM}/llvm-objdump", "-d", "--no-show-raw-insn", code_object], check=True, capture_output=True, text=True).stdout
    bad = {}
    for name, body in re.findall(r"^[0-9a-f]+ <(gi_\w+)>:\n(.*?)(?=^[0-9a-f]+ <|\Z)", asm, re.M | re.S):
        loops = len(re.findall(r"s_and_saveexec_b64[^\n]*\n(?:\s*s_nop[^\n]*\n)?\s*buffer_load", body))
        if loops:
            bad[name] = loops
    assert "<gi_prefill_fwd_i8>" in asm and not bad, bad
