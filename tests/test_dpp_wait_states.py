"""DPP operands in inline assembly.

On gfx950 an instruction that reads a vector register through DPP needs two
wait states after the instruction that wrote it.  The compiler inserts them for
its own instructions but does not look inside inline assembly, where it may
also place a register copy right in front.  So in the device assembly each
block that holds DPP instructions has to begin with its own wait states, and
to keep two between a write of its own and a DPP read of it, also where the
read follows the block.
"""
from __future__ import annotations

import glob
import os
import re
import shutil
import subprocess

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "msplat_amd")
SOURCES = sorted(p for p in glob.glob(os.path.join(PKG, "csrc", "*.hip")) if "_f32_dpp" in open(p).read())


def _registers(operand):
    m = re.match(r"v(\d+)$|v\[(\d+):(\d+)\]$", operand)
    if not m:
        return set()
    if m.group(1):
        return {int(m.group(1))}
    return set(range(int(m.group(2)), int(m.group(3)) + 1))


def _violations(lines):
    """DPP reads in one assembly block with fewer than two wait states behind
    them since the block's start or a write of the register."""
    bad = []
    waited, written = 0, {}    # wait states so far; register -> those at its write
    for line in lines:
        m = re.match(r"s_nop (\d+)", line)
        if m:
            waited += int(m.group(1)) + 1
            continue
        if line.startswith("v_"):
            ops = [o.strip() for o in line.split(None, 1)[1].split(",")]
            if "_dpp" in line:
                for r in _registers(ops[1]):
                    if waited - written.get(r, 0) < 2:
                        bad.append(line)
            for r in _registers(ops[0]):
                written[r] = waited + 1
        waited += 1
    return bad


def test_the_check_itself():
    add = "v_add_f32_dpp v1, v1, v1 row_shr:1 row_mask:0xf bank_mask:0xf"
    assert _violations([add]) == [add]
    assert _violations(["s_nop 0", add]) == [add]
    assert _violations(["s_nop 1", add]) == []
    assert _violations(["s_nop 1", add, add]) == [add]
    assert _violations(["s_nop 1", add, "v_mov_b32_e32 v2, v3", add]) == [add]
    assert _violations(["s_nop 1", add, "v_mov_b32_e32 v2, v3", "s_nop 0", add]) == []


@pytest.mark.parametrize("source", SOURCES, ids=os.path.basename)
def test_assembly_blocks_wait_before_dpp_reads(source):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if not (shutil.which(hipcc) and shutil.which("make")):
        pytest.skip("no hipcc")
    target = os.path.join("_build", os.path.basename(source)[:-4] + ".s")
    subprocess.check_call(["make", "-s", "-C", PKG, target], stderr=subprocess.DEVNULL)
    lines = [line.strip() for line in open(os.path.join(PKG, target))]
    blocks = 0
    for i, line in enumerate(lines):
        if line != ";;#ASMSTART":
            continue
        end = lines.index(";;#ASMEND", i)
        block = [x for x in lines[i + 1:end] if x]
        if not any("_dpp" in x for x in block):
            continue
        blocks += 1
        # the two instructions behind the block may read what it wrote
        behind = [x for x in lines[end + 1:end + 12] if re.match(r"[sv]_|ds_|global_|buffer_", x)][:2]
        assert not _violations(block + behind), (source, i, _violations(block + behind)[:4])
    assert blocks > 0
