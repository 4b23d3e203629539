"""The built engine's device code: a carry-in that a vector instruction wrote is
read two wait states later at the earliest. The compiler sees to that for its
own instructions, not for the inline assembly of fp_masks.h."""
import os
import re
import subprocess

import pytest

from fastpartitioner_amd import _native

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
CARRY = re.compile(r"v_(addc|subb|subbrev)_co_u32")


def _sgprs(op):
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", op)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.fullmatch(r"s(\d+)", op)
    return {int(m[1])} if m else {"vcc"} if op == "vcc" else set()


def _operands(text):
    return [x.strip() for x in re.findall(r"(?:[^,\[]|\[[^\]]*\])+", text)]


def _written(name, ops):
    """SGPRs a vector instruction writes."""
    if not name.startswith("v_") or not ops:
        return set()
    return _sgprs(ops[0]) | (_sgprs(ops[1]) if "_co_" in name and len(ops) > 1 else set())


def early_carries(lines):
    """(carry reads, the ones that come too early) of a disassembly."""
    kernel, before, reads, early = "", [], 0, []
    for line in lines:
        m = re.match(r"^[0-9a-f]+ <(.*)>:", line)
        if m:
            kernel, before = m[1], []
            continue
        m = re.match(r"^\s+([a-z_0-9]+)\s*(.*?)\s*(//.*)?$", line)
        if not m:
            continue
        name, ops = m[1], _operands(m[2])
        if CARRY.match(name):
            reads += 1
            carry, states = _sgprs(ops[-1]), 0
            for pname, pops in reversed(before):
                if states >= 2:
                    break
                if _written(pname, pops) & carry:
                    early.append((kernel, pname, pops, name, ops))
                    break
                states += 1 + (int(pops[0], 0) if pname == "s_nop" else 0)
        before = (before + [(name, ops)])[-3:]
    return reads, early


def test_the_check_finds_an_early_carry():
    text = ["0000 <k>:", "\tv_cmp_eq_u32_e64 s[0:1], s73, v3", "\tv_subbrev_co_u32_e64 v18, vcc, 0, v13, s[0:1]",
            "\tv_cmp_eq_u32_e64 s[2:3], s73, v3", "\ts_nop 1", "\tv_addc_co_u32_e64 v18, vcc, 0, v13, s[2:3]"]
    reads, early = early_carries(text)
    assert reads == 2 and len(early) == 1 and early[0][3] == "v_subbrev_co_u32_e64"


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_no_carry_comes_too_early(tmp_path):
    lib = tmp_path / "engine.so"
    lib.write_bytes(open(_native.ENGINE_LIB, "rb").read())
    subprocess.run([OBJDUMP, "--offloading", str(lib)], check=True, cwd=tmp_path, stdout=subprocess.DEVNULL)
    objects = [f for f in os.listdir(tmp_path) if "gfx950" in f]
    assert objects
    reads = 0
    for f in objects:
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", f], check=True, cwd=tmp_path, capture_output=True,
                              text=True).stdout
        n, early = early_carries(text.splitlines())
        reads += n
        assert not early, early[:5]
    assert reads > 500  # the masks' counts are among them
