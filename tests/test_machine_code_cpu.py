"""Wait states around the LDS DMA instructions, read from the gfx950 code in
the built library.

The kernels issue LDS DMA (global_load_lds_*, buffer_load_* ... lds) from
inline asm, where the compiler's hazard recogniser does not look, so the two
rules that it keeps for its own code are checked here on every one of them:
  * M0 (the LDS address) written by a scalar instruction: one wait state, that
    is one other instruction, before the DMA reads it;
  * a scalar register written by a vector instruction (v_readfirstlane_b32):
    five wait states before a vector memory instruction reads it.
"""

import os
import re
import shutil
import struct
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "jax-metallib_amd", "lib",
                   "libmk_kernels.so")
OBJDUMP = shutil.which("llvm-objdump", path="/opt/rocm/llvm/bin") or shutil.which("llvm-objdump")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects():
    """The gfx950 code objects of the library's offload bundles."""
    with open(LIB, "rb") as f:
        blob = f.read()
    out, at = [], blob.find(MAGIC)
    while at >= 0:
        entries, = struct.unpack_from("<Q", blob, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(entries):
            off, size, name = struct.unpack_from("<QQQ", blob, p)
            if b"gfx950" in blob[p + 24:p + 24 + name] and size:
                out.append(blob[at + off:at + off + size])
            p += 24 + name
        at = blob.find(MAGIC, at + 1)
    return out


def _states(line):
    """Wait states that an instruction stands for."""
    m = re.match(r"s_nop (\d+)", line)
    return int(m.group(1)) + 1 if m else 1


def _scalars(text):
    """The numbers of the scalar registers named in an operand list."""
    regs = set()
    for lo, hi, one in re.findall(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b", text):
        regs.update(range(int(lo), int(hi) + 1) if lo else (int(one),))
    return regs


def _faults(lines):
    """(LDS DMA instructions, those within a wait state too few)."""
    seen, bad = 0, []
    for i, line in enumerate(lines):
        if "_load_lds_" not in line and not (line.startswith("buffer_load") and line.endswith(" lds")):
            continue
        seen += 1
        reads = _scalars(line)
        states, j = 0, i - 1
        while j >= 0 and states < 5:
            prev = lines[j]
            op, _, operands = prev.partition(" ")
            target = operands.split(",")[0]
            if states < 1 and target == "m0":
                bad.append((prev, line))
            if op.startswith("v_") and target.startswith("s") and _scalars(target) & reads:
                bad.append((prev, line))
            if op == "s_endpgm" or prev.endswith(">:"):
                break
            states += _states(prev)
            j -= 1
    return seen, bad


def test_the_check_sees_a_missing_wait_state():
    dma = "global_load_lds_dwordx4 v[2:3], off"
    assert _faults(["s_mov_b32 m0, s4", dma])[1]
    assert not _faults(["s_mov_b32 m0, s4", "s_nop 0", dma])[1]
    based = "global_load_lds_dword v2, s[4:5]"
    assert _faults(["v_readfirstlane_b32 s5, v1", "s_nop 3", based])[1]
    assert not _faults(["v_readfirstlane_b32 s5, v1", "s_nop 4", based])[1]


@pytest.mark.skipif(OBJDUMP is None, reason="no llvm-objdump")
def test_lds_dma_keeps_its_wait_states(tmp_path):
    assert os.path.exists(LIB), "build the library first"
    total, bad = 0, []
    for i, code in enumerate(_code_objects()):
        path = tmp_path / f"{i}.co"
        path.write_bytes(code)
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--mcpu=gfx950", str(path)], check=True,
                              capture_output=True, text=True).stdout
        lines = [re.sub(r"\s*//.*", "", s).strip() for s in text.splitlines()]
        seen, faults = _faults([s for s in lines if s])
        total += seen
        bad += faults
    assert total > 100, "the library's LDS DMA was not found"
    assert not bad, f"{len(bad)} of {total} LDS DMA instructions too close, e.g. {bad[:3]}"
