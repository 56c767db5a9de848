"""Wait states of the written-out assembly in the reverse march (and in the lane
operations it shares with the step, fivonagi_amd/csrc/fv_lanes.h).  A DPP read of
a VGPR needs two wait states after the instruction that wrote it.  The compiler
sees neither the writes nor the DPP reads inside an asm block, so the blocks
have to hold the wait states themselves: whatever stands between a block and
what comes before or after it is not counted here."""
import os
import re
import shutil
import subprocess

import pytest

from fivonagi_amd import build

SRC = os.path.join(build.HERE, "csrc", "fv_adjoint_march.hip")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
NEEDED = 2


def vgprs(operand):
    m = re.match(r"^[-|]*v(?:(\d+)\b|\[(\d+):(\d+)\])", operand.strip())
    if not m:
        return []
    lo, hi = (m.group(1),) * 2 if m.group(1) else m.groups()[1:]
    return range(int(lo), int(hi) + 1)


def unguarded(asm):
    """DPP reads less than two wait states behind their operand's write, where
    one of the two is in an asm block."""
    bad = []
    block = 0              # the asm block we are in (0: the compiler's code)
    blocks = wait = 0      # wait states since the start of the block
    last = {}              # VGPR -> (block, wait state of its write, or left at its end)
    for line in asm.splitlines():
        if "#ASMSTART" in line:
            blocks += 1
            block, wait = blocks, 0
            continue
        if "#ASMEND" in line:
            last = {r: (b, wait - w) if b == block else (b, w) for r, (b, w) in last.items()}
            block = 0
            continue
        code = line.split(";")[0].strip()
        if not re.match(r"[vsgbd]\w*_", code) or code.endswith(":"):
            continue
        op, _, rest = code.partition(" ")
        if op == "s_nop":
            wait += int(rest, 0) + 1
            continue
        ops = rest.split(",")
        if op.startswith("v_"):
            if re.search(r"wave_sh|wave_ro|row_|quad_perm", rest):
                for r in vgprs(ops[1]):
                    b, w = last.get(r, (0, 0))
                    if not b and not block:
                        continue
                    have = wait - w if b == block else (w if b else 0) + (wait if block else 0)
                    if have < NEEDED:
                        bad.append((code, r, have))
            for r in vgprs(ops[0]):
                last[r] = (block, wait + 1 if block else 0)
        elif re.match(r"(global|flat|scratch|buffer)_load|ds_", op):
            for r in vgprs(ops[0]):        # (waited for by a counter)
                last.pop(r, None)
        wait += 1
    return bad


def test_the_check_finds_a_missing_wait():
    asm = "\n".join(["#ASMSTART", "v_mul_f32_e32 v1, v2, v2", "{}", "#ASMEND",
                     "v_mov_b32_dpp v3, v1 wave_shl:1 row_mask:0xf bank_mask:0xf"])
    assert unguarded(asm.format("")) and unguarded(asm.format("s_nop 0"))
    assert not unguarded(asm.format("s_nop 1"))
    assert list(vgprs("v[4:5]")) == [4, 5] and list(vgprs("-|v7|")) == [7]
    asm = "\n".join(["v_mul_f32_e32 v1, v2, v2", "#ASMSTART", "{}",
                     "v_add_f32_dpp v3, v1, v3 wave_shl:1 row_mask:0xf", "#ASMEND"])
    assert unguarded(asm.format("v_mul_f32_e32 v9, v8, v8"))
    assert not unguarded(asm.format("v_mul_f32_e32 v9, v8, v8\nv_mul_f32_e32 v7, v8, v8"))


@pytest.mark.skipif(shutil.which(HIPCC) is None, reason="needs hipcc")
def test_blocks_hold_their_wait_states(tmp_path):
    out = tmp_path / "march.s"
    flags = [f for f in build.HIPCC_FLAGS if f not in ("-shared", "-fPIC", "-pthread", "-Wall")]
    subprocess.run([HIPCC, *flags, "--cuda-device-only", "-S", SRC, "-o", str(out)], check=True,
                   stderr=subprocess.DEVNULL)
    asm = out.read_text()
    assert asm.count("#ASMSTART") > 10
    assert unguarded(asm) == []
