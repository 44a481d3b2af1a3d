"""The build's check for spills in front of a join's exec restore (CPU only): it finds the two that
one build of the fused kernel had, and the built library has none."""
import os
import subprocess
import sys

import pytest

import isa_check

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "sph-exa-nnet_amd", "lib", "libnnet_mi355x.so")

# the end of the loop that loads a net87 particle's abundances, as that build had it; {0}: in front
# of the restore, {1}: behind it
BLOCK = """
0000000000001000 <kernel>:
\ts_and_saveexec_b64 s[0:1], vcc                              // 000000001000: BE80206A
\ts_cbranch_execz 5                                           // 000000001004: BF880005 <kernel+0x1c>
\tv_mov_b32_e32 v2, 0                                         // 000000001008: 7E040280
\tds_write_b64 v2, v[4:5]                                     // 00000000100C: D89A0000 00000402
\ts_andn2_b64 exec, exec, s[26:27]                            // 000000001014: 89FE1A7E
\ts_cbranch_execnz 65532                                      // 000000001018: BF89FFFC <kernel+0xc>
\tv_writelane_b32 v255, s40, 57                               // 00000000101C: D28A00FF 00017228
\ts_mov_b32 s38, 0                                            // 000000001024: BEA60080
{0}\ts_or_b64 exec, exec, s[0:1]                                 // 000000001038: 87FE007E
{1}\ts_endpgm                                                    // 00000000104C: BF810000
"""
SPILLS = ("\tscratch_store_dwordx2 off, v[154:155], off offset:32        // 00000000{:X}: DC744020 007F9A00\n"
          "\tscratch_store_dwordx2 off, v[152:153], off offset:24        // 00000000{:X}: DC744018 007F9800\n")


@pytest.mark.parametrize("front", [True, False])
def test_spills_in_front_of_the_restore(front):
    text = BLOCK.format(SPILLS.format(0x1028, 0x1030), "") if front else BLOCK.format("", SPILLS.format(0x103c, 0x1044))
    found, joins = isa_check.findings(text)
    assert joins == 1  # the branch on an empty mask and the loop's end lead to the same block
    assert [a for _, a, _ in found] == ([0x1028, 0x1030] if front else [])


def test_else_branch_and_lane_moves():
    # the other side of an if / else restores with a saveexec form; register-to-lane moves do not
    # depend on the mask; a narrower branch that starts right away is no restore
    head = "0000000000000ffc <kernel>:\n\ts_and_saveexec_b64 s[0:1], vcc   // 000000000FFC: BE80206A\n"
    head += "\ts_cbranch_execz 1     // 000000001000: BF880001 <kernel+0xc>\n\ts_nop 0       // 000000001004: BF800000\n"
    tail = "\ts_endpgm               // 000000001018: BF810000\n"
    for first, mask, hits in (("v_mov_b32_e32 v1, v2", "s_andn2_saveexec_b64 s[0:1], s[54:55]", 1),
                              ("v_mov_b32_e32 v1, v2", "s_or_saveexec_b64 s[0:1], s[54:55]", 1),
                              ("v_readlane_b32 s4, v255, 3", "s_or_b64 exec, exec, s[0:1]", 0),
                              ("v_mov_b32_e32 v1, v2", "s_and_saveexec_b64 s[0:1], vcc", 0)):
        text = head + f"\t{first}      // 000000001008: 7E020302\n\t{mask}      // 000000001010: 87FE007E\n" + tail
        assert len(isa_check.findings(text)[0]) == hits, (first, mask)


def test_branch_that_is_never_taken():
    # the compiler writes some branches that are never taken as branches on an empty mask: the mask
    # was not narrowed for them, and what they lead to is ordinary code in front of a restore
    text = """
0000000000001000 <kernel>:
{0}\ts_nop 0                                                     // 000000001004: BF800000
\ts_cbranch_execz 1                                           // 000000001008: BF880001 <kernel+0x10>
\ts_branch 2                                                  // 00000000100C: BF820002 <kernel+0x18>
\tv_mul_f64 v[18:19], v[4:5], s[0:1]                          // 000000001010: D2810012 00000104
\ts_or_b64 exec, exec, s[2:3]                                 // 000000001018: 87FE027E
\ts_endpgm                                                    // 00000000101C: BF810000
"""
    for before, hits in (("", 0), ("\ts_and_saveexec_b64 s[2:3], vcc        // 000000001000: BE82206A\n", 1),
                         ("\ts_or_b64 exec, exec, s[2:3]            // 000000001000: 87FE027E\n", 0)):
        assert len(isa_check.findings(text.format(before))[0]) == hits, before


def test_built_library_has_none():
    if not os.path.exists(LIB) or not os.path.exists(isa_check.OBJDUMP):
        pytest.skip("library not built or no llvm-objdump")
    found, joins = isa_check.findings(isa_check.disassemble(LIB))
    assert joins > 1000 and not found, found[:10]
    r = subprocess.run([sys.executable, isa_check.__file__, LIB], capture_output=True, text=True)
    assert r.returncode == 0 and "0 misplaced" in r.stdout
