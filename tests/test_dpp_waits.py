"""Wait states before lane moves, in the built library's own gfx950 code.

A DPP move may read a vector register no sooner than two wait states after a
vector instruction wrote it.  The compiler places them after its own
instructions, but it does not look into assembly blocks, and the field products
(csrc/mont_asm.hpp) are one block each whose results the lane layouts of
csrc/curve_split.hpp move between lanes: only the order of the moves (limb 0
first, the block writes limbs 7 and 8 last) keeps the distance.  This test looks
at every such move of the library that was built, so that a change of the moves,
the blocks or the compiler's order cannot break it unseen.
"""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "cuda-zkml_amd", "libzkml_gpu.so")
OBJDUMP = shutil.which("llvm-objdump", path="/opt/rocm/llvm/bin:" + os.environ.get("PATH", ""))
WAITS = 2


def vgprs(operand):
    m = re.fullmatch(r"v(?:(\d+)|\[(\d+):(\d+)\])", operand)
    if not m:
        return range(0)
    return range(int(m[1]), int(m[1]) + 1) if m[1] else range(int(m[2]), int(m[3]) + 1)


def close_reads(lines):
    """(DPP moves, those that read a register within WAITS wait states of its
    write) of a disassembly."""
    moves, close = 0, []
    recent = []  # (registers written, wait states of the instruction, text), the last few
    for line in lines:
        text = line.split("//")[0].strip()
        if not text or text.endswith(":"):
            continue
        op, _, rest = text.partition(" ")
        args = re.split(r",\s*|\s+", rest.strip())
        if "_dpp" in op:
            moves += 1
            waits = 0
            for written, states, writer in reversed(recent):
                if waits >= WAITS:
                    break
                if any(r in written for r in vgprs(args[1])):
                    close.append((writer, text))
                    break
                waits += states
        recent.append((vgprs(args[0]) if op.startswith("v_") else range(0),
                       int(args[0], 0) + 1 if op == "s_nop" else 1, text))
        del recent[:-WAITS]
    return moves, close


def test_close_reads_are_found():
    write, move = "\tv_and_b32_e32 v9, 0x1fffffff, v54", "\tv_mov_b32_dpp v1, v9 quad_perm:[1,0,3,2] row_mask:0xf"
    other = "\tv_add_u32_e32 v2, v3, v4"
    assert len(close_reads([write, move])[1]) == 1
    assert len(close_reads([write, other, move])[1]) == 1
    assert len(close_reads([write, "\ts_nop 0", move])[1]) == 1
    assert close_reads([write, "\ts_nop 1", move]) == (1, [])
    assert close_reads([write, other, other, move]) == (1, [])
    assert len(close_reads(["\tv_mad_u64_u32 v[8:9], vcc, v1, v2, v[8:9]", move])[1]) == 1


@pytest.mark.skipif(not OBJDUMP, reason="no llvm-objdump")
def test_lane_moves_wait_for_their_operands(tmp_path):
    assert os.path.exists(LIB), "build the library first"
    shutil.copy(LIB, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    objects = sorted(p for p in tmp_path.iterdir() if p.name.endswith("gfx950"))
    assert objects
    moves = 0
    for obj in objects:
        asm = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", str(obj)], check=True,
                             capture_output=True, text=True).stdout
        n, close = close_reads(asm.splitlines())
        moves += n
        assert not close, (obj.name, len(close), close[:3])
    assert moves > 1000  # the lane layouts are there
