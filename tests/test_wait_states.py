"""Wait states that gfx9 leaves to the program, looked for in the built library's own instructions.  The compiler puts
them in by itself, but not inside an inline instruction block and not in front of one."""
import glob
import os
import re
import shutil
import subprocess

import pytest

from tiny_llm_amd.kernels import library

OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
AFTER_M0 = 1          # wait states from a scalar write of M0 to a load into LDS
AFTER_VALU = 5        # ... from a vector instruction's scalar result to a memory instruction that reads it


def scalars(operand):
    """The scalar registers an operand names: s4, s[4:7], m0, vcc."""
    m = re.fullmatch(r"s(\d+)|s\[(\d+):(\d+)\]", operand)
    if m:
        first, last = (m[1], m[1]) if m[1] else (m[2], m[3])
        return {f"s{i}" for i in range(int(first), int(last) + 1)}
    return {operand} if operand in ("m0", "vcc") else set()


def short_waits(lines):
    """(what is too close, the load) for every load into LDS in a listing."""
    found, recent = [], []                # recent: (wait states since, scalars written, by a vector instruction, text)
    for line in lines:
        m = re.match(r"\s+([a-z]\w+)(?:\s+(.*?))?\s*(?://.*)?$", line)
        if not m:
            continue
        name, operands = m[1], [o.strip() for o in re.split(r",(?![^\[]*\])", m[2] or "")]
        words = [w for o in operands for w in o.split()]
        if "_load_lds_" in name or words[-1:] == ["lds"]:
            read = set().union(*(scalars(w) for w in words)) if words else set()
            for since, written, vector, text in recent:
                if "m0" in written and since < AFTER_M0 or vector and written & read and since < AFTER_VALU:
                    found.append((text, line.strip()))
        states = int(operands[0], 0) + 1 if name == "s_nop" else 1
        recent = [(s + states, w, v, t) for s, w, v, t in recent if s + states < AFTER_VALU]
        vector = name.startswith("v_")
        written = set().union(*(scalars(o) for o in operands[:2 if vector else 1])) if operands else set()
        if written and name.startswith(("s_", "v_")):
            recent.append((0, written, vector, line.strip()))
    return found


def test_the_rules_find_what_they_are_for():
    m0, load = "\ts_mov_b32 m0, s2", "\tbuffer_load_dwordx4 v94, s[4:7], s14 offen lds // 0000"
    assert short_waits([m0, load]) and not short_waits([m0, "\ts_nop 0", load])
    assert short_waits(["\ts_add_u32 m0, s2, 4", "\tglobal_load_lds_dwordx4 v[0:1], off"])
    lane = "\tv_readfirstlane_b32 s6, v1"
    assert short_waits([lane, "\ts_nop 3", load]) and not short_waits([lane, "\ts_nop 4", load])
    assert not short_waits(["\tv_readfirstlane_b32 s8, v1", load])


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_loads_into_lds_keep_their_wait_states(tmp_path):
    lib = shutil.copy(library.find_or_build(verbose=False), tmp_path / "kernels.so")
    subprocess.run([OBJDUMP, "--offloading", str(lib)], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    loads, short = 0, []
    for part in sorted(glob.glob(str(tmp_path / f"*{library.ARCH}*"))):
        text = subprocess.run([OBJDUMP, "-d", part], check=True, capture_output=True, text=True).stdout.splitlines()
        loads += sum(" lds" in line.split("//")[0] or "_load_lds_" in line for line in text)
        short += short_waits(text)
    assert loads > 0
    assert not short, f"{len(short)} of {loads} loads, the first: {short[0]}"
