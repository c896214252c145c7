"""Wait states that the compiler cannot see to: its hazard pass does not look
inside inline asm, so the built gfx950 code is disassembled and checked."""
import os
import re
import shutil
import subprocess

import pytest

from kb_nano_amd._build import LIB_PATH

OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"


def _sgprs(text):
    regs = set()
    for lo, hi, one in re.findall(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b", text):
        regs |= {int(one)} if one else set(range(int(lo), int(hi) + 1))
    return regs


def _functions(tmp_path):
    """(name, [(instruction, operands), ...]) of every gfx950 function in the library."""
    so = shutil.copy(LIB_PATH, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", str(so)], cwd=tmp_path, check=True, capture_output=True)
    objects = sorted(p for p in tmp_path.iterdir() if p.name.endswith("gfx950"))
    assert objects
    for obj in objects:
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(obj)], check=True, capture_output=True,
                              text=True).stdout
        name, code = None, []
        for line in text.splitlines():
            if m := re.match(r"[0-9a-f]+ <(.+)>:$", line):
                if code:
                    yield name, code
                name, code = m.group(1), []
            elif m := re.match(r"\s+(\w+)\s*(.*?)\s*(?://.*)?$", line):
                code.append(m.groups())
        if code:
            yield name, code


def hazards(code):
    """The loads and stores of one function that come too early: an LDS load
    right after a scalar write of M0 (one wait state needed), and a vector
    memory instruction less than five wait states after a vector instruction
    wrote an SGPR that it reads; these are the gaps that the gfx950 compiler
    leaves around its own instructions."""
    found, at, m0, valu, lds_loads = [], 0, -9, {}, 0
    for op, args in code:
        if op == "s_nop":
            at += int(args) + 1
            continue
        at += 1
        dst = args.split(",")[0]
        if op.startswith(("buffer_", "global_", "flat_", "scratch_")):
            if args.endswith(" lds"):
                lds_loads += 1
                if at - m0 < 2:
                    found.append(("M0", op, args))
            found += [("SGPR", op, args) for r in _sgprs(args) if at - valu.get(r, -9) < 6]
        elif op.startswith("s_") and dst == "m0":
            m0 = at
        elif op.startswith(("v_readfirstlane", "v_readlane", "v_cmp")):
            valu.update(dict.fromkeys(_sgprs(dst), at))
    return found, lds_loads


def test_the_check_sees_both_hazards():
    load = ("buffer_load_dword", "v0, s[0:3], s8 offen lds")
    assert hazards([("s_add_u32", "m0, s4, 0x100"), load]) == ([("M0", *load)], 1)
    assert hazards([("s_mov_b32", "m0, s4"), ("s_nop", "0"), load]) == ([], 1)
    assert hazards([("s_mov_b32", "m0, s4"), ("v_mov_b32_e32", "v1, v2"), load]) == ([], 1)
    for gap, bad in ((3, True), (4, False)):
        assert bool(hazards([("v_readfirstlane_b32", "s2, v1"), ("s_nop", str(gap)), load])[0]) is bad


def test_built_kernels_keep_the_wait_states(tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    loads = 0
    for name, code in _functions(tmp_path):
        found, n = hazards(code)
        loads += n
        assert not found, f"{name}: {len(found)} of {n} LDS loads, e.g. {found[0]}"
    assert loads > 1000   # the GEMM kernels' direct loads were seen
