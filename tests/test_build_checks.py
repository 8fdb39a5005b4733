"""The check that the build makes of the accumulators of inline-assembly MFMAs (eisen_amd/csrc/check_agpr_loops.py)."""
import importlib.util
import os

import pytest

from tests.conftest import ROOT

_spec = importlib.util.spec_from_file_location("check_agpr_loops", os.path.join(ROOT, "eisen_amd", "csrc", "check_agpr_loops.py"))
agpr = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(agpr)

LISTING = """\t.text
some_kernelILi128E:                     ; @some
; %bb.0:
\tv_accvgpr_write_b32 a0, 0
.LBB0_1:                                ; =>This Loop
\tv_mov_b32_e32 v9, 0
.LBB0_2:                                ;   a[0:15] in a comment is not a use
\tds_read_b128 v[0:3], v8
\t;;#ASMSTART
\ts_nop 1
\tv_mfma_f32_32x32x16_bf16 a[0:15], v[0:3], v[4:7], a[0:15]
\t;;#ASMEND
\tv_add_u32_e32 v8, 16, v8
\ts_cbranch_scc1 .LBB0_4
; %bb.3:
\ts_branch .LBB0_2
.LBB0_5:                                ; not behind the loop: the path of a wave without tiles
\tv_accvgpr_write_b32 a0, 0
.LBB0_4:
\tv_mov_b32_e32 v10, 0
\t;;#ASMSTART
\ts_nop 15
\ts_nop 7
\t;;#ASMEND
\tv_accvgpr_read_b32 v0, a0
\ts_cbranch_vccnz .LBB0_1
\ts_endpgm
.Lfunc_end0:
"""


def test_the_sound_listing_passes():
    assert agpr.check(LISTING, "some_kernel", 1) == []


@pytest.mark.parametrize("where,line,message", [
    ("\tds_read_b128 v[0:3], v8\n", "\tv_accvgpr_read_b32 v11, a3\n", "in the loop"),
    ("\tv_add_u32_e32 v8, 16, v8\n", "\tv_accvgpr_mov_b32 a20, a3\n", "in the loop"),
    ("\tv_add_u32_e32 v8, 16, v8\n", "\tscratch_store_dword off, v3, off\n", "scratch access"),
    ("\tv_add_u32_e32 v8, 16, v8\n", "\tv_mfma_f32_32x32x2_f32 a[16:31], v0, v1, a[16:31]\n", "in the loop"),
    ("\tv_mov_b32_e32 v10, 0\n", "\tv_accvgpr_read_b32 v11, a3\n", "before the wait states"),
])
def test_a_planted_use_of_an_accumulator_is_found(where, line, message):
    assert any(message in m for m in agpr.check(LISTING.replace(where, where + line), "some_kernel", 1))


def test_missing_wait_states_loops_and_kernels_are_found():
    assert any("no wait states" in m for m in agpr.check(LISTING.replace("s_nop 15", "s_nop 3").replace("v_accvgpr_read_b32 v0, a0", "s_nop 0"), "some_kernel", 1))
    assert any("no loop" in m for m in agpr.check(LISTING.replace("s_branch .LBB0_2", "s_nop 0").replace("s_cbranch_vccnz .LBB0_1", "s_nop 0"), "some_kernel", 1))
    assert any("expected 2" in m for m in agpr.check(LISTING, "some_kernel", 2))
