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
    if operand in ("vcc", "vcc_lo", "vcc_hi"):
        return {"vcc": {"vcc_lo", "vcc_hi"}}.get(operand, {operand})
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    if m:
        return set(range(int(m.group(1)), int(m.group(2)) + 1))
    m = re.fullmatch(r"s(\d+)", operand)
    return {int(m.group(1))} if m else set()


class _Instruction:
    def __init__(self, text, comment, address):
        self.text = text
        self.op, _, rest = text.partition(" ")
        self.operands = [o.strip().split(" ")[0] for o in rest.split(",")] if rest else []
        m = re.search(r"\b([0-9A-F]{8,}):", comment)
        self.address = int(m.group(1), 16) if m else address
        m = re.search(r"<\w+\+0x([0-9a-f]+)>", comment)
        self.target = int(m.group(1), 16) if m else None        # from the function's start
        self.ends = self.op in ("s_branch", "s_endpgm", "s_setpc_b64")
        self.width = int(self.operands[0], 0) + 1 if self.op == "s_nop" else 1
        written = self.operands[:1]
        if re.search(r"_co_|^v_div_scale|^v_mad_[ui]64", self.op):
            written = self.operands[:2]
        self.by_vector = set().union(*map(_scalars, written)) if self.op.startswith("v_") and written else set()
        self.by_scalar = set()
        if re.match(r"s_(mov|add|sub|mul|lsh|ash|and|or|xor|min|max|cselect)", self.op) and written:
            self.by_scalar = _scalars(written[0])


def _functions(lines):
    """name -> [instructions], with the long jumps (s_getpc, s_add, s_addc, s_setpc) resolved."""
    functions, name, start = {}, "", 0
    for line in lines:
        m = re.match(r"^([0-9a-f]+) <(\w+)>:", line)
        if m:
            start, name = int(m.group(1), 16), m.group(2)
            functions[name] = (start, [])
            continue
        text, _, comment = line.partition("//")
        text = text.strip()
        if name and re.match(r"^[a-z]", text):
            functions[name][1].append(_Instruction(text, comment, start + len(functions[name][1])))
    for start, code in functions.values():
        for at, ins in enumerate(code):
            if ins.target is not None:
                ins.target += start
            if ins.op != "s_setpc_b64":
                continue
            low, offset = min(_scalars(ins.operands[0])), None
            for back in range(at - 1, max(at - 12, 0), -1):
                prior = code[back]
                if prior.op in ("s_add_u32", "s_sub_u32") and prior.operands[0] == f"s{low}" and offset is None:
                    offset = int(prior.operands[2], 0) * (1 if prior.op == "s_add_u32" else -1)
                if prior.op == "s_getpc_b64" and prior.operands[0] == ins.operands[0] and offset is not None:
                    ins.target = code[back + 1].address + ((offset + 2 ** 31) % 2 ** 32 - 2 ** 31)
                    break
            assert ins.target is not None, f"a jump that is not understood: {ins.text}"
    return {name: code for name, (_, code) in functions.items()}


def _too_early(lines):
    """(function, instruction) of every memory operation too close behind such a write, on any way
    that leads to it."""
    found = []
    for name, code in _functions(lines).items():
        at_address = {ins.address: i for i, ins in enumerate(code)}
        jumps = {}
        for i, ins in enumerate(code):
            if ins.target is not None and ins.op.startswith(("s_branch", "s_cbranch", "s_setpc")):
                jumps.setdefault(at_address[ins.target], []).append(i)

        def early(i, used, states):
            before = jumps.get(i, []) + ([i - 1] if i > 0 and not code[i - 1].ends else [])
            for j in before:
                ins = code[j]
                if ins.by_vector & used:
                    return True
                rest = used - ins.by_scalar     # (replaced by a scalar instruction: no distance to keep)
                if rest and states + ins.width < WAIT_STATES and early(j, rest, states + ins.width):
                    return True
            return False

        for i, ins in enumerate(code):
            if re.match(r"(global|buffer|scratch|flat)_", ins.op):
                used = set().union(*map(_scalars, ins.operands)) if ins.operands else set()
                if used and early(i, used, 0):
                    found.append((name, ins.text))
    return found


def test_the_check_sees_a_load_that_comes_too_early():
    code = ["0000 <k>:", "  v_readlane_b32 s4, v254, 58", "  v_readlane_b32 s5, v254, 59",
            "  global_load_dwordx4 v[74:77], v130, s[4:5]"]
    assert _too_early(code) == [("k", "global_load_dwordx4 v[74:77], v130, s[4:5]")]
    assert _too_early(code[:3] + ["  s_nop 4"] + code[3:]) == []
    assert _too_early(code[:3] + ["  s_nop 3"] + code[3:]) != []
    assert _too_early(code[:3] + ["  s_mov_b64 s[4:5], s[8:9]"] + code[3:]) == []
    # ... and by way of a jump, a short one or a long one
    around = ["0000 <k>:", "  s_cbranch_scc0 3 // 00000000: <k+0x14>", "  s_nop 4 // 00000004:",
              "  v_readlane_b32 s4, v254, 58 // 00000008:", "  s_branch 1 // 0000000C: <k+0x18>",
              "  s_endpgm // 00000010:", "  s_nop 4 // 00000014:",
              "  global_load_dwordx4 v[74:77], v130, s[4:5] // 00000018:"]
    assert len(_too_early(around)) == 1
    assert _too_early(around[:4] + ["  s_endpgm // 0000000C:"] + around[5:]) == []
    far = around[:4] + ["  s_getpc_b64 s[10:11] // 0000000C:", "  s_add_u32 s10, s10, 0x30 // 00000010:",
                        "  s_addc_u32 s11, s11, 0 // 00000018:", "  s_setpc_b64 s[10:11] // 0000001C:",
                        "  s_nop 4 // 00000020:", "  global_load_dwordx4 v[74:77], v130, s[4:5] // 00000040:"]
    assert len(_too_early([line.replace("+0x14", "+0x20") for line in far])) == 1


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
