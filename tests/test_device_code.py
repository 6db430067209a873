"""The check of the built device code (spike_amd/devcode.py): it finds the block it is for, lets
the forms around it pass, and passes the library that is built."""
import pytest

from spike_amd import abi, devcode

# a divergent branch over [0x0108, 0x0110), joined at 0x0110
_LISTING = """
co:\tfile format elf64-amdgpu

Disassembly of section .text:

0000000000000100 <kernel>:
\ts_and_saveexec_b64 s[2:3], vcc                             // 000000000100: BE82206A
\ts_cbranch_execz 3                                          // 000000000104: BF880003 <kernel+0x10>
\tv_add_u32_e32 v1, v2, v3                                   // 000000000108: 68020702
%s
\tv_add_u32_e32 v4, v4, v4                                   // 000000000130: 68080908
"""
_OR = "s_or_b64 exec, exec, s[2:3]"


def _block(*instructions):
    """The instructions from the joined block's start on."""
    return _LISTING % "\n".join(f"\t{i:<58} // {0x110 + 4 * k:012X}: 00000000" for k, i in enumerate(instructions))


@pytest.mark.parametrize("instructions", [
    ("s_mov_b32 s4, s5", "v_mov_b32_e32 v47, v107", _OR),
    ("v_mov_b32_e32 v47, v107", _OR),
    ("v_accvgpr_write_b32 a3, v1", "s_nop 1", _OR),
    ("s_waitcnt vmcnt(0)", "scratch_store_dword off, v3, off", _OR)])
def test_copy_before_the_mask_is_restored(instructions):
    found = devcode.copies_before_exec_restore(_block(*instructions))
    assert [(f, len(c)) for f, _, c in found] == [("kernel", 1)]


@pytest.mark.parametrize("instructions", [
    (_OR, "v_mov_b32_e32 v47, v107"),
    ("s_mov_b32 s4, s5", _OR, "v_mov_b32_e32 v47, v107"),
    ("v_readlane_b32 s4, v47, 3", _OR),
    ("v_mov_b32_e32 v47, v107", "v_add_u32_e32 v1, v2, v3", _OR),          # a block of the branch's own
    ("v_mov_b32_e32 v47, v107", "s_and_saveexec_b64 s[6:7], vcc", _OR)])
def test_forms_that_are_right(instructions):
    assert devcode.copies_before_exec_restore(_block(*instructions)) == []


def test_built_library():
    assert devcode.check(abi.LIB_PATH) > 100
