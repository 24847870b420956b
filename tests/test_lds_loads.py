"""The wait states around loads straight into LDS, in the built kernels. They are written in assembly, whose inside the compiler's own
pass over such hazards does not see: a scalar write of m0 needs an instruction or an s_nop between it and the load that reads it, and
a vector instruction that writes the load's scalar address needs five."""
import os
import re
import shutil
import subprocess

import pytest

from mini_llm_amd import build

OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"


def scalar_registers(operand):
    span = re.match(r"s\[(\d+):(\d+)\]$", operand)
    if span:
        return set(range(int(span[1]), int(span[2]) + 1))
    one = re.match(r"s(\d+)$", operand)
    return {int(one[1])} if one else set()


def hazards(lines):
    """(loads into LDS, those too close behind a write of m0, those too close behind a vector write of their address)"""
    loads, m0, address = 0, [], []
    for i, line in enumerate(lines):
        if not re.match(r"(global|buffer)_load_lds_", line):
            continue
        loads += 1
        read = set().union(*(scalar_registers(o) for o in re.split(r"[ ,]+", line)[1:]))
        waited = 0
        for before in reversed(lines[max(0, i - 5):i]):
            if before.startswith("s_nop"):
                waited += int(before.split()[1], 0) + 1
                continue
            op, *operands = re.split(r"[ ,]+", before)
            if waited < 1 and op.startswith("s_") and operands[:1] == ["m0"]:
                m0.append(f"{before} > {line}")
            written = operands[:2 if "_co_" in op or "div_scale" in op else 1]          # (a second result is a carry)
            if waited < 5 and op.startswith("v_") and any(scalar_registers(o) & read for o in written):
                address.append(f"{before} > {line}")
            waited += 1
    return loads, m0, address


def test_the_check_sees_the_hazards():
    load = "global_load_lds_dwordx4 v11, s[4:5]"
    assert hazards(["s_mov_b32 m0, s58", load]) == (1, [f"s_mov_b32 m0, s58 > {load}"], [])
    assert hazards(["s_mov_b32 m0, s58", "s_nop 0", load]) == (1, [], [])
    assert hazards(["s_mov_b32 m0, s58", "v_add_u32_e32 v1, v2, v3", load]) == (1, [], [])
    assert hazards(["v_readfirstlane_b32 s5, v0", "s_mov_b32 m0, s58", "s_nop 0", load])[2] != []
    assert hazards(["v_readfirstlane_b32 s5, v0", "s_nop 2", "s_mov_b32 m0, s58", "s_nop 0", load]) == (1, [], [])
    assert hazards(["v_mov_b32_e32 v0, s5", "s_mov_b32 m0, s58", "s_nop 0", load]) == (1, [], [])
    assert hazards(["v_add_co_u32_e64 v0, s[4:5], v1, v2", "s_mov_b32 m0, s58", "s_nop 0", load])[2] != []
    assert hazards(["v_readfirstlane_b32 s6, v0", "s_mov_b32 m0, s58", "s_nop 0", load]) == (1, [], [])


@pytest.mark.parametrize("name", ["gemm_bf16", "gemm_f32", "attention"])
def test_loads_into_lds_wait_for_their_scalars(name, tmp_path):
    if not os.path.isfile(OBJDUMP):
        pytest.skip("no llvm-objdump on this machine")
    if not build.is_current(name):
        build.build_library(name)
    library = shutil.copy(build.lib_path(name), tmp_path)
    subprocess.run([OBJDUMP, "--offloading", library], cwd=tmp_path, check=True, capture_output=True)
    code = [f for f in os.listdir(tmp_path) if f.endswith(build.GPU_ARCH)]
    assert len(code) == 1, os.listdir(tmp_path)
    text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", code[0]], cwd=tmp_path, check=True, capture_output=True,
                          text=True).stdout
    loads, m0, address = hazards([line.split("//")[0].strip() for line in text.splitlines()])
    assert loads > 0
    assert not m0 and not address, (len(m0), len(address), loads, (m0 + address)[:3])
