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


@pytest.fixture(scope="module")
def code_objects(tmp_path_factory):
    """The assembler's lines for each of the library's device code objects, by name."""
    if not os.path.exists(OBJDUMP) or not os.path.exists(LIB):
        pytest.skip("no llvm-objdump, or the library is not built")
    at = tmp_path_factory.mktemp("code")
    lib = shutil.copy(LIB, at / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", str(lib)], cwd=at, check=True, stdout=subprocess.DEVNULL)
    return {name: subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", name], cwd=at, check=True, stdout=subprocess.PIPE, text=True).stdout.splitlines()
            for name in sorted(os.listdir(at)) if name.endswith("gfx950")}


def test_the_rule_is_recognised():
    after = ["s_mov_b32 m0, s9", "s_nop 0", "buffer_load_dwordx4 v1, s[4:7], s2 offen lds"]
    for first in ("v_readfirstlane_b32 s2, v0", "v_readlane_b32 s6, v0, 3"):
        assert len(hazards([first] + after)[0]) == 1
        assert hazards([first, after[0], "s_nop 3", after[2]])[0] == []
    assert hazards(["v_readfirstlane_b32 s3, v0"] + after)[0] == []
    assert len(hazards([after[0], after[2]])[0]) == 1


def test_loads_into_lds_wait_for_their_scalars(code_objects):
    loads = 0
    for name, lines in code_objects.items():
        if not any(" lds" in line for line in lines):
            continue
        bad, n = hazards(lines)
        assert not bad, f"{len(bad)} of {n} in {name}, the first: {bad[0]}"
        loads += n
    assert loads > 100, "the blocked kernels' loads were not found"


def test_the_blocked_kernel_stores_through_the_caches(code_objects):
    """Rows whose length is no multiple of 128 bytes share their lines between workgroups: stores with the non-temporal hint
    write such a line in pieces (up to 1.6 times the call's time)."""
    kernel, stores = "", 0
    for line in (line for lines in code_objects.values() for line in lines):
        text = line.split("//")[0].strip()
        if text.endswith(">:"):
            kernel = text
        elif "block_kernel" in kernel and text.startswith("buffer_store"):
            assert not re.search(r"\b(nt|sc0|sc1)\b", text), (kernel, text)
            stores += 1
    assert stores > 30 * 16, "the blocked kernels' stores were not found"
