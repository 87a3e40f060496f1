"""The build's check of device assembly: a vector register spilled ahead of
the instruction that gives a block its lanes back is reported, the same spill
behind it is not."""

import os
import runpy

import pytest

CHECK = runpy.run_path(os.path.join(os.path.dirname(__file__), "..", "psychopath_amd", "csrc", "check_spills.py"))

BLOCK = """_Z6kernelv:                            ; @_Z6kernelv
; %bb.0:
	s_and_saveexec_b64 s[0:1], vcc
	s_cbranch_execz .LBB3_2
; %bb.1:
	global_load_dword v4, v[6:7], off
	{inside}
.LBB3_2:
	{head}
	{restore}
	{behind}
	s_endpgm
.Lfunc_end3:
"""
SPILL = "scratch_store_dword off, v4, off offset:28 ; 4-byte Folded Spill"


def asm(inside="s_nop 0", head="s_nop 0", restore="s_or_b64 exec, exec, s[0:1]", behind="s_nop 0"):
    return BLOCK.format(inside=inside, head=head, restore=restore, behind=behind)


@pytest.mark.parametrize("head,restore", [
    (SPILL, "s_or_b64 exec, exec, s[0:1]"),
    ("s_waitcnt vmcnt(0)\n\tv_mov_b32_e32 v9, 0\n\t" + SPILL, "s_or_b64 exec, exec, s[0:1]"),
    (SPILL, "s_or_saveexec_b64 s[2:3], s[0:1]"),
    ("v_accvgpr_write_b32 a3, v4", "s_or_b64 exec, exec, s[0:1]"),
])
def test_early_spill_is_found(head, restore):
    found = CHECK["early_spills"](asm(head=head, restore=restore))
    assert [(k, label) for k, label, _ in found] == [("_Z6kernelv", ".LBB3_2")]


@pytest.mark.parametrize("text", [
    asm(),
    asm(inside=SPILL),                                   # the branch's own lanes, on its side
    asm(behind=SPILL),                                   # all lanes are back
    asm(head="v_add_f32_e32 v4, v5, v4\n\t" + SPILL),    # a block with work of its own before the next join
    asm(head=SPILL, restore="s_and_saveexec_b64 s[2:3], vcc"),
])
def test_other_spills_are_not(text):
    assert CHECK["early_spills"](text) == []


def test_exit_status(tmp_path):
    good, bad = tmp_path / "good.s", tmp_path / "bad.s"
    good.write_text(asm())
    bad.write_text(asm(head=SPILL))
    assert CHECK["main"]([str(good)]) == 0
    assert CHECK["main"]([str(good), str(bad)]) == 1
