"""The batched prefill's masked multiply-adds write exec by inline asm
(fma_below in csrc/prefill.hip).  On gfx950 a vector instruction's write of
exec wants 4 wait states before a lane read or write and 5 before a DPP
operand; the compiler inserts them for its own writes only.  Here the device
assembly of that source, built with the library's flags, is read for every
such write."""
import os
import re
import shutil
import subprocess

import pytest

from conftest import PKG

LANE = re.compile(r"v_(readlane|readfirstlane|writelane|permlane)")
DPP = re.compile(r"\b(quad_perm|row_shl|row_shr|row_ror|row_bcast|row_newbcast|row_mirror|row_half_mirror|wave_shl|wave_shr|wave_rol|wave_ror)\b|_dpp\b")


def exec_hazards(text):
    """(the v_cmpx instructions, the lines that follow one too early).  Every
    instruction is a wait state, s_nop N is N + 1; a branch or the code's end
    within them counts as too early (what follows is not in the text)."""
    writes, bad, since = 0, [], 99
    for line in text.splitlines():
        ins = line.split(";")[0].strip()
        if not ins or ins.startswith(".") or ins.endswith(":"):
            continue
        if ins.startswith("v_cmpx"):
            writes, since = writes + 1, 0
            continue
        if (since < 4 and (LANE.match(ins) or re.match(r"s_(c?branch|setpc|swappc|endpgm)", ins))) or (since < 5 and DPP.search(ins)):
            bad.append(line.strip())
        nop = re.match(r"s_nop (\d+)", ins)
        since += int(nop.group(1)) + 1 if nop else 1
    return writes, bad


@pytest.mark.parametrize("between,early", [
    ("", True), ("s_nop 3", False), ("s_nop 2", True), ("s_add_i32 s1, s1, 1\n s_nop 1\n s_mov_b64 exec, -1", False),
    ("v_fma_f64 v[0:1], s[0:1], v[2:3], v[0:1]\n s_mov_b64 exec, -1\n s_nop 0", True)])
def test_the_check_sees_a_lane_write_too_early(between, early):
    asm = f"  v_cmpx_gt_u32_e32 vcc, s1, v1 ; comment\n {between}\n.Llabel:\n  v_writelane_b32 v7, s3, 2\n"
    assert exec_hazards(asm) == (1, ["v_writelane_b32 v7, s3, 2"] if early else [])
    dpp = f"  v_cmpx_gt_u32_e32 vcc, s1, v1\n {between}\n  v_add_u32_dpp v7, v7, v8 row_shr:1 row_mask:0xf\n"
    assert len(exec_hazards(dpp)[1]) == 1   # 4 wait states are one short


def test_prefill_exec_writes_settle():
    if not (shutil.which("make") and os.path.exists("/opt/rocm/bin/hipcc")):
        pytest.skip("no hipcc")
    subprocess.run(["make", "-C", PKG, "build/prefill.s"], check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    with open(os.path.join(PKG, "build", "prefill.s")) as f:
        writes, bad = exec_hazards(f.read())
    assert writes >= 3 * 16   # three instances, 16 tokens each
    assert not bad, bad[:5]
