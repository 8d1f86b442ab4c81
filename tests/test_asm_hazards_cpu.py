"""The LDS-DMA issue paths obey the gfx9 wait-state rules that the compiler cannot add itself.

The kernels issue ``global_load_lds_dwordx4`` from inline asm (so that the compiler's
wait-count pass does not serialise ring reads behind it), and the hazard recognizer does not
look inside inline asm. Two rules then fall to the source, and this test checks them on the
device assembly of every kernel source, built here for gfx950 (no GPU needed):

* a vector-ALU write of an SGPR (``v_readfirstlane_b32`` of a DMA base address, a compare's
  lane mask, a carry-out) needs 5 wait states before a memory instruction reads that SGPR -- a
  stale base reads a wild address;
* a scalar write of M0 needs 1 wait state before an LDS DMA reads M0.

The check follows the control flow: each kernel's assembly is split into basic blocks (labels,
branches, ``s_endpgm``), and from every memory instruction it walks back over every path into
it -- fall-through, branch targets and loop back-edges -- until the wait states add up.
"""

from __future__ import annotations

import glob
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "mini-sglang_amd"))
import build  # noqa: E402  (mini-sglang_amd/build.py: the flags the library is built with)
from asm_check import find_hazards, functions, open_dma_statements  # noqa: E402

HIPCC = build.HIPCC
SOURCES = sorted(glob.glob(os.path.join(build.CSRC, "*.hip")))


def _device_asm(src: str, out_dir: str) -> str:
    out = os.path.join(out_dir, os.path.basename(src) + ".s")
    cmd = [HIPCC, *build.FLAGS, *build.SOURCE_FLAGS.get(os.path.basename(src), []), "--cuda-device-only", "-S",
           src, "-o", out]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    with open(out) as f:
        return f.read()


def test_checker_catches_a_readfirstlane_feeding_a_dma():
    asm = """
        .type k,@function
k:
        v_readfirstlane_b32 s1, v3
        v_readfirstlane_b32 s0, v2
        s_mov_b32 m0, s6
        global_load_lds_dwordx4 v253, s[0:1]
        s_nop 4
        s_add_i32 m0, s6, 0x1000
        s_nop 0
        global_load_lds_dwordx4 v252, s[0:1]
        s_endpgm
.Lfunc_end0:
    """
    sgpr, m0 = find_hazards(asm)
    assert len(sgpr) == 1 and "v_readfirstlane_b32 s0" in sgpr[0][1]
    assert len(m0) == 1 and "s_mov_b32 m0" in m0[0][1]


def test_checker_follows_loop_back_edges_and_branches():
    """A readfirstlane at the bottom of a loop feeds the DMA at its top (the back-edge), a compare's
    lane mask and a carry-out feed DMAs across a branch; the same code with enough wait states on
    every path is clean."""
    bad = """
        .type k,@function
k:
        s_mov_b32 s4, 0
.LBB0_1:
        s_mov_b32 m0, s5
        s_nop 0
        global_load_lds_dwordx4 v10, s[0:1]
        v_mfma_f32_16x16x32_bf16 v[20:23], v[2:5], v[6:9], v[20:23]
        s_add_i32 s4, s4, 1
        s_cmp_lt_i32 s4, 8
        v_readfirstlane_b32 s0, v12
        s_cbranch_scc1 .LBB0_1
        v_cmp_gt_i32_e64 s[8:9], v1, v2
        s_cbranch_vccz .LBB0_3
        s_nop 1
.LBB0_3:
        global_load_dword v3, v4, s[8:9]
        v_add_co_u32_e64 v5, s[10:11], v6, v7
        s_branch .LBB0_4
.LBB0_4:
        global_load_dword v3, v4, s[10:11]
        s_endpgm
.Lfunc_end0:
    """
    sgpr, m0 = find_hazards(bad)
    got = sorted(h[1].split()[0] + " -> " + h[2].split()[-1] for h in sgpr)
    assert got == ["v_add_co_u32_e64 -> s[10:11]", "v_cmp_gt_i32_e64 -> s[8:9]", "v_readfirstlane_b32 -> s[0:1]"]
    assert not m0
    good = bad.replace("s_cbranch_scc1 .LBB0_1", "s_nop 4\n        s_cbranch_scc1 .LBB0_1").replace(
        "s_cbranch_vccz .LBB0_3\n        s_nop 1", "s_nop 4\n        s_cbranch_vccz .LBB0_3\n        s_nop 1").replace(
        "v_add_co_u32_e64 v5, s[10:11], v6, v7", "v_add_co_u32_e64 v5, s[10:11], v6, v7\n        s_nop 4")
    assert find_hazards(good) == ([], [])


def test_checker_counts_the_last_write_only():
    """A spilled address restored with readlanes and then rebuilt by scalar adds is read by the DMA
    from the scalar writes: no hazard. Rebuilding only its low half leaves the readlane of the high
    half as the last write: a hazard."""
    asm = """
        .type k,@function
k:
        v_readlane_b32 s4, v239, 10
        s_add_u32 s4, s4, s8
        v_readlane_b32 s5, v239, 11
        s_addc_u32 s5, s5, s3
        s_mov_b32 m0, s3
        s_nop 0
        global_load_lds_dwordx4 v4, s[4:5]
        s_endpgm
.Lfunc_end0:
    """
    assert find_hazards(asm) == ([], [])
    half = asm.replace("s_addc_u32 s5, s5, s3", "s_nop 0")
    sgpr, m0 = find_hazards(half)
    assert len(sgpr) == 1 and "v_readlane_b32 s5" in sgpr[0][1] and not m0


def test_checker_m0_across_a_branch():
    asm = """
        .type k,@function
k:
        s_cbranch_execz .LBB0_2
        s_mov_b32 m0, s3
.LBB0_2:
        global_load_lds_dwordx4 v1, s[0:1]
        s_endpgm
.Lfunc_end0:
    """
    sgpr, m0 = find_hazards(asm)
    assert not sgpr and len(m0) == 1


def test_checker_catches_a_dma_statement_without_waits():
    asm = """
        ;;#ASMSTART
        s_nop 0
        global_load_lds_dwordx4 v10, s[0:1]
        ;;#ASMEND
        ;;#ASMSTART
        s_nop 4
        global_load_lds_dwordx4 v10, s[0:1] nt
        ;;#ASMEND
        ;;#ASMSTART
        s_nop 0
        global_load_lds_dwordx4 v[10:11], off
        ;;#ASMEND
    """
    assert open_dma_statements(asm) == [["s_nop 0", "global_load_lds_dwordx4 v10, s[0:1]"]]


def test_build_fails_on_a_hazard():
    asm = """
        .type k,@function
k:
        v_readlane_b32 s1, v3, 4
        s_nop 0
        global_load_lds_dwordx4 v253, s[0:1]
        s_endpgm
.Lfunc_end0:
    """
    with pytest.raises(RuntimeError, match="x.hip: .*v_readlane_b32 s1"):
        build.check_assembly("x.hip", asm)
    build.check_assembly("x.hip", asm.replace("s_nop 0", "s_nop 4"))


@pytest.mark.skipif(shutil.which(HIPCC) is None and not os.path.exists(HIPCC), reason="hipcc not available")
@pytest.mark.parametrize("src", [os.path.basename(s) for s in SOURCES])
def test_no_dma_hazards(src, tmp_path):
    path = os.path.join(build.CSRC, src)
    asm = _device_asm(path, str(tmp_path))
    with open(path) as f:
        has_kernels = "__global__" in f.read()
    assert bool(functions(asm)) == has_kernels, "kernel symbols not found in the device assembly"
    sgpr, m0 = find_hazards(asm)
    if src.startswith("mla_decode"):  # (the prefill kernel's loads share one wait, spread over a step's slots)
        assert not open_dma_statements(asm), "a DMA statement does not wait for its own base"
    assert not sgpr, f"VALU-written SGPR read by a memory instruction too early: {sgpr[:3]}"
    assert not m0, f"M0 written right before an LDS DMA: {m0[:3]}"
