"""Wait states ahead of the loads from memory straight into LDS, in the gfx950
code of the built library.

Such a load takes its LDS address from M0 and its range from four SGPRs.  The
hardware does not hold it back for either: a scalar write of M0 needs one wait
state before it, a vector instruction's write of one of the SGPRs five.  The
compiler puts them in for instructions that it knows, not for those written as
inline assembly, which is how the prefill kernels issue these loads."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from slm_testlib import load_product

P = load_product()
OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")
INSTR = re.compile(r"^\s+([a-z]\w+)\s*(.*?)\s*//")


def regs(operand):
    """SGPRs that an operand names."""
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.fullmatch(r"s(\d+)", operand)
    return {int(m[1])} if m else set()


def lds_loads_without_their_waits(lines):
    """(number of loads into LDS, those that follow a write too closely)."""
    found, bad, before = 0, [], []  # before: (op, first operand, wait states it gives)
    for ln in lines:
        m = INSTR.match(ln)
        if not m:
            if ln.rstrip().endswith(">:"):
                before = []
            continue
        op, args = m[1], [a.strip() for a in m[2].split(",")]
        if op.startswith("buffer_load") and args[-1].split()[-1] == "lds":
            found += 1
            # operands: voffset, descriptor, soffset and flags
            need, waited = regs(args[1]), 0
            for bop, bdst in reversed(before):
                if bop == "s_nop":
                    waited += int(bdst, 0) + 1
                    continue
                if bdst == "m0" and waited < 1:
                    bad.append(f"{bop} {bdst}, ... {ln.strip()}")
                if bop.startswith("v_") and regs(bdst) & need and waited < 5:
                    bad.append(f"{bop} {bdst}, ... {ln.strip()}")
                waited += 1
                if waited >= 5:
                    break
        before = (before + [(op, args[0])])[-8:]
    return found, bad


@pytest.fixture(scope="module")
def listing(tmp_path_factory):
    if not OBJDUMP.exists():
        pytest.skip("llvm-objdump is not installed")
    d = tmp_path_factory.mktemp("code")
    lib = d / "lib.so"
    shutil.copy(P.LIB_PATH, lib)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=d)
    text = ""
    for obj in sorted(d.glob("*gfx950")):
        text += subprocess.run([OBJDUMP, "-d", obj], check=True, capture_output=True,
                               text=True).stdout
    return text.splitlines()


def test_loads_into_lds_wait_for_their_address(listing):
    found, bad = lds_loads_without_their_waits(listing)
    assert found >= 14, "the split prefill's forms stage their tiles with such loads"
    assert not bad, (len(bad), bad[:4])


def test_the_check_sees_a_missing_wait():
    load = "\tbuffer_load_dwordx4 v80, s[4:7], 0 offen lds // 0: E0"
    for ahead, missing in (
            (["\ts_mov_b32 m0, s65 // 0"], 1),
            (["\ts_add_i32 m0, s4, 0x1000 // 0", "\ts_nop 0 // 0"], 0),
            (["\ts_mov_b32 m0, s65 // 0", "\tv_add_u32_e32 v1, v2, v3 // 0"], 0),
            (["\tv_readfirstlane_b32 s6, v1 // 0", "\ts_nop 3 // 0"], 1),
            (["\tv_readfirstlane_b32 s6, v1 // 0", "\ts_nop 4 // 0"], 0),
            (["\tv_readfirstlane_b32 s8, v1 // 0"], 0)):
        found, bad = lds_loads_without_their_waits(ahead + [load])
        assert found == 1 and len(bad) == missing, ahead
