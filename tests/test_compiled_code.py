"""The compiled kernels: the search of their assembly for register copies that miss lanes
(oceano_amd/check_code.py), and what they spill."""
import glob
import os
import re
import shutil
import subprocess

import pytest

from oceano_amd.build import LIB
from oceano_amd.check_code import partial_copies

# the block at fault, as the compiler wrote it, and its surroundings
SIDE = """_Zkernel:
; %bb.0:
\tv_mov_b32_e32 v1, v0
\ts_and_saveexec_b64 s[0:1], s[20:21]
\ts_xor_b64 s[0:1], exec, s[0:1]
\ts_cbranch_execz .LBB0_2
; %bb.1:
\tv_add_f64 v[184:185], v[184:185], v[2:3]
.LBB0_2:
HEAD; %bb.3:
\tv_add_f64 v[184:185], v[184:185], v[4:5]
.LBB0_4:
\ts_or_b64 exec, exec, s[0:1]
\ts_endpgm
.Lfunc_end0:
"""
COPIES = "\tv_accvgpr_write_b32 a38, v184\n\tv_accvgpr_write_b32 a39, v185\n"
SCALAR = "\ts_mov_b64 s[72:73], s[54:55]\n"
READ_LANE = "\tv_readlane_b32 s56, v251, 17\n"
ON = "\ts_or_saveexec_b64 s[0:1], s[0:1]\n"
OFF = "\ts_xor_b64 exec, exec, s[0:1]\n\ts_cbranch_execz .LBB0_4\n"
ON_OFF = "\ts_andn2_saveexec_b64 s[0:1], s[0:1]\n\ts_cbranch_execz .LBB0_4\n"


@pytest.mark.parametrize("head,found", [
    (COPIES + SCALAR + ON + OFF, True),
    (COPIES + SCALAR + ON_OFF, True),
    ("\tv_mov_b64_e32 v[8:9], v[184:185]\n" + SCALAR + ON + OFF, True),
    ("\tscratch_store_dwordx2 off, v[184:185], off\n" + ON + OFF, True),
    (SCALAR + ON + COPIES + OFF, False),
    (SCALAR + READ_LANE + ON_OFF, False),
    ("\tv_cmp_lt_i32_e32 vcc, 1, v46\n" + ON_OFF, False),
])
def test_else_block(head, found):
    got = partial_copies(SIDE.replace("HEAD", head).splitlines(True))
    assert [g[:2] for g in got] == ([("_Zkernel", ".LBB0_2")] if found else [])


@pytest.mark.parametrize("first,found", [("", True), ("\tv_add_f64 v[8:9], v[2:3], v[4:5]\n", False)])
def test_block_entered_from_above(first, found):
    """without the skip a block follows the side that ran: its own work may stand there"""
    text = SIDE.replace("HEAD", first + COPIES + SCALAR + ON + OFF)
    text = text.replace("\ts_cbranch_execz .LBB0_2\n", "")
    got = partial_copies(text.replace(".LBB0_2:", "; %bb.2:").splitlines(True))
    assert [g[:2] for g in got] == ([("_Zkernel", "%bb.2")] if found else [])


def test_end_of_a_branch():
    text = SIDE.replace("HEAD", ON + OFF).replace(".LBB0_4:\n", ".LBB0_4:\n" + COPIES + SCALAR)
    assert [g[:2] for g in partial_copies(text.splitlines(True))] == [("_Zkernel", ".LBB0_4")]
    # skips are a kernel's own
    other = text.replace("_Zkernel", "_Zother").replace("s_cbranch_execz .LBB0_4", "s_nop 0")
    got = partial_copies((text + other).splitlines(True))
    assert [g[:2] for g in got] == [("_Zkernel", ".LBB0_4")]


OBJDUMP, READELF = ("/opt/rocm/llvm/bin/llvm-" + t for t in ("objdump", "readelf"))


def _registers(tmp_path):
    """{kernel: (vector registers it uses, those it spills)}, from the built library's metadata"""
    shutil.copy(LIB, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", os.path.basename(LIB)], cwd=tmp_path, check=True,
                   stdout=subprocess.DEVNULL)
    out = {}
    for part in glob.glob(str(tmp_path / "*gfx950")):
        notes = subprocess.run([READELF, "--notes", part], check=True, stdout=subprocess.PIPE,
                               text=True).stdout
        for kernel in notes.split("  - .agpr_count")[1:]:
            name = re.search(r"\.name:\s+(\S+)", kernel).group(1)
            out[name] = tuple(int(re.search(r"\.vgpr_%scount:\s+(\d+)" % what, kernel).group(1))
                              for what in ("", "spill_"))
    return out


tools = pytest.mark.skipif(not (os.path.exists(OBJDUMP) and os.path.exists(READELF)),
                           reason="no ROCm tools")


@tools
def test_fp64_stage_kernels_keep_their_registers(tmp_path):
    """FP64 stage, M^-1 L, L and additive kernels at p = 3 (every terms type, paired or not): the few
    registers of a loop's bookkeeping may be spilled, not its work"""
    spilled = {k: v[1] for k, v in _registers(tmp_path).items()
               if re.search(r"k_stage(_pair|_ark_pair)?ILi3E(Lb[01]E)?d", k)}
    assert len(spilled) >= 20
    assert max(spilled.values()) <= 4, {k: v for k, v in spilled.items() if v > 4}


@tools
@pytest.mark.parametrize("kernel,most,spills", [
    (r"k_stageILi3ELb1Ef\w*OpArgsELi0E", 256, 0),     # viscous stage: two waves per SIMD
    (r"k_stageILi2ELb1Ef\w*OpArgsELi0E", 128, 0),     # four
    (r"k_stage_pairILi2EfLb[01]ELb0ELi0E", 128, 0),
    (r"k_height_jacobiILi[12]E", 128, 0),
    (r"k_height_jacobiILi3E", 256, 0),
    (r"k_depth_deferredILi3E", 256, 0)])
def test_kernels_with_the_sweeps_keep_their_waves(tmp_path, kernel, most, spills):
    """FP32 kernels that hold the FP64 sweeps of dry cells, and the split path's depth solve"""
    got = {k: v for k, v in _registers(tmp_path).items() if re.search(kernel, k)}
    assert got
    assert all(v[0] <= most and v[1] <= spills for v in got.values()), got
