"""Wait states the built kernels owe the hardware, read from the library's own assembly.

The compiler inserts the wait states CDNA asks for between its own instructions, but
not around inline asm, which the attention kernels issue their row DMAs with. Checked
on every instruction of the built library:

* a VMEM instruction reads no SGPR that a VALU instruction (``v_readlane``, ``v_cmp``, ...)
  wrote fewer than five wait states before it: it could read the old value, a wrong address;
* an LDS DMA has one wait state between it and a scalar write of M0.

CPU only (``llvm-objdump`` of the ROCm toolchain that built the library).
"""

import os
import re
import shutil
import subprocess

import pytest

from sparse_attn_sharedkv_amd import _lib

OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
VMEM = ("global_", "buffer_", "scratch_", "flat_")


def _regs(operand):
    """The scalar registers an operand names: numbers, and 'vcc' / 'm0'."""
    out = set()
    for a, b in re.findall(r"\bs\[(\d+):(\d+)\]", operand):
        out |= set(range(int(a), int(b) + 1))
    out |= {int(a) for a in re.findall(r"\bs(\d+)\b", operand)}
    out |= set(re.findall(r"\b(vcc|m0)", operand))
    return out


def _parse(line):
    """(mnemonic, operands) of a line of disassembly or compiler output, or None."""
    text = line.split("//")[0].split(";")[0].strip()
    if not text or text.endswith(":") or text.startswith((".", "<")):
        return None
    op, _, rest = text.partition(" ")
    return op, [x.strip() for x in rest.split(",")] if rest else []


def short_waits(lines):
    """The instructions of ``lines`` that follow a register write they depend on too soon."""
    bad, window = [], []  # window: the latest instructions, newest last
    for line in lines:
        ins = _parse(line)
        if ins is None:
            continue
        op, args = ins
        if op.startswith(VMEM):
            reads, states = set().union(*map(_regs, args)), 0
            for prev, pargs in reversed(window):
                if states >= 5:
                    break
                if prev.startswith("v_") and pargs:
                    dst = _regs(pargs[0])
                    if ("_co_" in prev or "div_scale" in prev) and len(pargs) > 1:
                        dst |= _regs(pargs[1])
                    if dst & reads:
                        bad.append(f"{states} wait states: {prev} {', '.join(pargs)} -> {line.strip()}")
                        break
                if states == 0 and "_lds_" in op and pargs and _regs(pargs[0]) & {"m0"}:
                    bad.append(f"no wait state: {prev} {', '.join(pargs)} -> {line.strip()}")
                    break
                states += int(pargs[0], 0) + 1 if prev == "s_nop" else 1
        window = [] if op in ("s_branch", "s_endpgm", "s_setpc_b64") else window[-6:] + [ins]
    return bad


@pytest.mark.parametrize("code, n", [
    ("v_readlane_b32 s5, v1, 0\ns_mov_b32 m0, s9\ns_nop 0\n"
     "global_load_lds_dwordx4 v2, s[4:5] sc0 nt", 1),        # 2 wait states of 5
    ("v_readlane_b32 s5, v1, 0\ns_mov_b32 m0, s9\ns_nop 3\n"
     "global_load_lds_dwordx4 v2, s[4:5] sc0 nt", 0),
    ("v_readlane_b32 s5, v1, 0\ns_mov_b32 m0, s9\ns_mov_b64 s[6:7], s[4:5]\n"
     "global_load_lds_dwordx4 v2, s[6:7] sc0 nt", 0),        # a scalar copy
    ("s_mov_b32 m0, s9\nglobal_load_lds_dwordx4 v[2:3], off", 1),
    ("v_cmp_eq_u32_e64 s[2:3], v0, v1\nglobal_load_dword v1, v0, s[2:3]", 1),
    ("v_cmp_eq_u32_e64 s[2:3], v0, v1\ns_nop 4\nglobal_load_dword v1, v0, s[2:3]", 0),
])
def test_the_reader_finds_short_waits(code, n):
    assert len(short_waits(code.split("\n"))) == n


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="llvm-objdump not found")
def test_built_kernels_keep_their_wait_states(tmp_path):
    lib = shutil.copy(_lib.LIB_PATH, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True,
                   capture_output=True)
    images = [f for f in os.listdir(tmp_path) if "gfx950" in f]
    assert images, "no gfx950 code in the library"
    dmas, bad = 0, []
    for f in images:
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", f], cwd=tmp_path, check=True,
                              capture_output=True, text=True).stdout
        dmas += text.count("global_load_lds_")
        bad += short_waits(text.split("\n"))
    assert dmas > 1000, "the attention kernels' row DMAs were not found"
    assert not bad, f"{len(bad)} instructions, the first:\n" + "\n".join(bad[:5])
