"""Wait states behind scalar registers, in the code that was built: a vector memory operation may
read a scalar register that a vector instruction wrote only five wait states later.  The compiler
keeps that distance in what it emits itself, but it does not look into inline assembly, and the
GEMM kernels' loads are inline: every memory operation of the built objects is checked."""
from __future__ import annotations

import re
import shutil
import subprocess
from pathlib import Path

import pytest

from vkernels_amd import build as vk_build

LLVM = Path("/opt/rocm/llvm/bin")
WAIT_STATES = 5


def _scalars(operand):
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    if m:
        return set(range(int(m.group(1)), int(m.group(2)) + 1))
    m = re.fullmatch(r"s(\d+)", operand)
    return {int(m.group(1))} if m else set()


def _too_early(lines):
    """(function, instruction) of every memory operation too close behind such a write."""
    found, name, history = [], "", []
    for line in lines:
        m = re.match(r"^[0-9a-f]+ <(\w+)>:", line)
        if m:
            name, history = m.group(1), []
            continue
        text = line.split("//")[0].strip()
        if not re.match(r"^[a-z]", text):
            continue
        op, _, rest = text.partition(" ")
        operands = [o.strip().split(" ")[0] for o in rest.split(",")] if rest else []
        if re.match(r"(global|buffer|scratch|flat)_", op):
            used = set().union(*map(_scalars, operands)) if operands else set()
            states = 0
            for written, width in reversed(history):
                if states >= WAIT_STATES:
                    break
                if written & used:
                    found.append((name, text))
                    break
                states += width
        width = int(operands[0], 0) + 1 if op == "s_nop" else 1
        if re.match(r"s_(mov|add|sub|mul|lsh|ash|and|or|xor|min|max|cselect)", op) and operands:
            for written, _ in history:  # (replaced by a scalar instruction: no distance to keep)
                written -= _scalars(operands[0])
        history.append((_scalars(operands[0]) if op.startswith("v_") and operands else set(), width))
        history = history[-WAIT_STATES:]
    return found


def test_the_check_sees_a_load_that_comes_too_early():
    code = ["0000 <k>:", "  v_readlane_b32 s4, v254, 58", "  v_readlane_b32 s5, v254, 59",
            "  global_load_dwordx4 v[74:77], v130, s[4:5]"]
    assert _too_early(code) == [("k", "global_load_dwordx4 v[74:77], v130, s[4:5]")]
    assert _too_early(code[:3] + ["  s_nop 4"] + code[3:]) == []
    assert _too_early(code[:3] + ["  s_nop 3"] + code[3:]) != []
    assert _too_early(code[:3] + ["  s_mov_b64 s[4:5], s[8:9]"] + code[3:]) == []


@pytest.mark.parametrize("unit", ["moe_prefill", "moe_gemm"])
def test_no_memory_operation_reads_a_scalar_too_early(unit, tmp_path):
    obj = vk_build.OBJ / f"{unit}.o"
    tools = [LLVM / n for n in ("llvm-objcopy", "clang-offload-bundler", "llvm-objdump")]
    if not obj.is_file() or not all(shutil.which(str(t)) for t in tools):
        pytest.skip("no object of this unit, or no LLVM tools")
    bundle, code = tmp_path / "bundle", tmp_path / "code"
    subprocess.run([tools[0], f"--dump-section=.hip_fatbin={bundle}", obj, tmp_path / "copy.o"], check=True)
    subprocess.run([tools[1], "--unbundle", "--type=o", f"--input={bundle}", f"--output={code}",
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
    dump = subprocess.run([tools[2], "-d", "--no-show-raw-insn", code], check=True, capture_output=True, text=True).stdout
    assert dump.count("v_mfma") > 1000
    early = _too_early(dump.splitlines())
    assert not early, f"{len(early)}, the first: {early[0]}"
