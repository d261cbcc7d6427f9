"""The library's own device code, read as the assembler prints it: rules of the instruction set that the compiler keeps
for its own instructions but not for those inside inline assembly.  No device needed."""
import os
import re
import shutil
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "meganeura_amd", "libmgn_hip.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def scalars(operand):
    """The scalar registers of one printed operand: s7, s[4:7], m0, vcc."""
    r = re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    if r:
        return {f"s{i}" for i in range(int(r[1]), int(r[2]) + 1)}
    return {operand} if re.fullmatch(r"s\d+|m0|vcc", operand) else set()


def hazards(lines):
    """Loads into LDS that read a scalar register less than five wait states after the vector unit wrote it, or M0 with none
    after a scalar write (an instruction is one state, s_nop n is n + 1)."""
    bad, loads, window = [], 0, []  # window: (text, name, what the first operand names, wait states)
    for line in lines:
        text = line.split("//")[0].strip()
        if not text or text.endswith(":"):
            window = [] if text.endswith(">:") else window
            continue
        name, _, rest = text.partition(" ")
        ops = [o for o in re.split(r"[,\s]+", rest.strip()) if o]
        if name.startswith("buffer_load") and ops[-1] == "lds":
            loads += 1
            read = set().union(*(scalars(o) for o in ops))
            states = 0
            for was, wname, wrote, n in reversed(window):
                if states == 0 and wname.startswith("s_") and "m0" in wrote:
                    bad.append((was, text))
                if states < 5 and wname.startswith("v_") and wrote & read:
                    bad.append((was, text))
                states += n
        window.append((text, name, scalars(ops[0]) if ops else set(), int(ops[0], 0) + 1 if name == "s_nop" else 1))
        window = window[-8:]
    return bad, loads


def test_the_rule_is_recognised():
    after = ["s_mov_b32 m0, s9", "s_nop 0", "buffer_load_dwordx4 v1, s[4:7], s2 offen lds"]
    for first in ("v_readfirstlane_b32 s2, v0", "v_readlane_b32 s6, v0, 3"):
        assert len(hazards([first] + after)[0]) == 1
        assert hazards([first, after[0], "s_nop 3", after[2]])[0] == []
    assert hazards(["v_readfirstlane_b32 s3, v0"] + after)[0] == []
    assert len(hazards([after[0], after[2]])[0]) == 1


def test_loads_into_lds_wait_for_their_scalars(tmp_path):
    if not os.path.exists(OBJDUMP) or not os.path.exists(LIB):
        pytest.skip("no llvm-objdump, or the library is not built")
    lib = shutil.copy(LIB, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", str(lib)], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    loads = 0
    for name in sorted(os.listdir(tmp_path)):
        if not name.endswith("gfx950"):
            continue
        out = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", name], cwd=tmp_path, check=True, stdout=subprocess.PIPE, text=True).stdout
        if " lds " not in out:
            continue
        bad, n = hazards(out.splitlines())
        assert not bad, f"{len(bad)} of {n} in {name}, the first: {bad[0]}"
        loads += n
    assert loads > 100, "the blocked kernels' loads were not found"
