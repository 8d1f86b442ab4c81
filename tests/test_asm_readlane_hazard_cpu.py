"""No v_readfirstlane / v_readlane reads a vector register in the wait state after a vector-ALU write of it.

gfx940 and later need one wait state between a vector-ALU write of a VGPR and a lane read of it. The
compiler's hazard recognizer adds it for its own instructions but does not look inside inline assembly, where
the kernels read DMA base addresses back to scalar registers; a base read too early is the register's old
value, and the DMA then loads from another row or a wild address. Checked on the device assembly of every
kernel source, over every control-flow path (no GPU needed).
"""

from __future__ import annotations

import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import test_asm_hazards_cpu as asm_check  # noqa: E402
from asm_check import find_lane_read_hazards  # noqa: E402


def test_checker_catches_a_lane_read_right_after_the_write():
    asm = """
        .type k,@function
k:
        v_lshl_add_u64 v[70:71], v[70:71], 0, s[38:39]
        v_readfirstlane_b32 s6, v70
        v_readfirstlane_b32 s7, v71
        v_add_u32_e32 v3, v1, v2
        s_nop 0
        v_readfirstlane_b32 s8, v3
        v_mov_b32_e32 v4, v5
        s_cbranch_scc0 .LBB0_2
.LBB0_2:
        v_readlane_b32 s9, v4, 3
        v_permlane32_swap_b32 v8, v9
        v_readfirstlane_b32 s9, v9
        s_endpgm
.Lfunc_end0:
    """
    assert [line for _, _, line in find_lane_read_hazards(asm)] == ["v_readfirstlane_b32 s6, v70",
                                                                    "v_readfirstlane_b32 s9, v9"]


@pytest.mark.skipif(not os.path.exists(asm_check.HIPCC), reason="needs hipcc")
@pytest.mark.parametrize("src", [os.path.basename(s) for s in asm_check.SOURCES])
def test_no_lane_read_hazards(src, tmp_path):
    asm = asm_check._device_asm(os.path.join(asm_check.build.CSRC, src), str(tmp_path))
    hazards = find_lane_read_hazards(asm)
    assert not hazards, f"{len(hazards)} lane reads of a register written by the instruction before: {hazards[:3]}"
