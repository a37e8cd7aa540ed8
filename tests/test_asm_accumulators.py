"""The check of matrix instructions in asm statements (moonep_amd/asm_waits.py), on pieces of assembly and
on what the compiler makes of the wide GEMM kernels."""

import pytest

from moonep_amd import asm_waits, build

MUL = "v_mfma_f32_16x16x32_bf16 a[0:3], v[4:7], v[8:11], a[0:3]"


def _asm(text):
    return (";;#ASMSTART", text, ";;#ASMEND")


def _faults(*lines):
    body = "\n".join(line if line.endswith(":") else f"\t{line}" for line in lines)
    return asm_waits.check(f"gemm_k:                                 ; @gemm_k\n{body}\n\ts_endpgm\n.Lfunc_end0:\n"
                           "amdhsa.kernels:\n  - .agpr_count: 4\n    .name:           gemm_k\n    .vgpr_spill_count: 0\n")[0]


@pytest.mark.parametrize("lines", [
    ("v_mov_b32 v4, v1", "s_nop 1", *_asm(MUL)),
    ("v_mov_b32 v4, v1", "s_mov_b32 s0, s1", "v_mov_b32 v1, v2", *_asm(MUL)),
    (*_asm(MUL), *_asm("v_accvgpr_read_b32 v1, a[0]")),
    ("v_mov_b32 v12, v1", *_asm(MUL)),
    # the loop's last write is two slots from its first matrix instruction; one behind the loop is not on its way
    (".LBB0_1:", "s_nop 0", *_asm(MUL), "v_mov_b32 v4, v1", "s_cbranch_scc1 .LBB0_1", "v_mov_b32 v5, v1"),
    # what follows an unconditional branch in the listing is not what follows it
    ("v_mov_b32 v4, v1", "s_branch .LBB0_2", ".LBB0_1:", *_asm(MUL), "s_endpgm", ".LBB0_2:", "s_nop 0", "s_branch .LBB0_1"),
    ("v_accvgpr_write_b32 a0, v1", "v_mfma_f32_16x16x32_bf16 a[0:3], v[4:7], v[8:11], a[0:3]"),   # the compiler's own
])
def test_right(lines):
    assert _faults(*lines) == []


@pytest.mark.parametrize("lines", [
    ("v_mov_b32 v4, v1", *_asm(MUL)),
    ("v_mov_b32 v11, v1", "s_mov_b32 s0, s1", *_asm(MUL)),
    ("v_mov_b32 v11, v1", "s_nop 0", *_asm(MUL)),
    (".LBB0_1:", *_asm(MUL), "v_mov_b32 v4, v1", "s_cbranch_scc1 .LBB0_1"),
    (".LBB0_1:", *_asm(MUL), "s_nop 3", "v_mov_b32 v8, v1", "s_branch .LBB0_1"),
    (*_asm(MUL), "v_accvgpr_read_b32 v1, a2"),
    ("v_accvgpr_mov_b32 a200, a7", "s_nop 3", *_asm(MUL)),
])
def test_wrong(lines):
    faults = _faults(*lines)
    assert len(faults) == 1 and "line" in faults[0]


def test_the_wide_kernels_as_they_are_compiled(tmp_path):
    path = str(tmp_path / "wide.s")
    build.gemm_assembly(path, source="gemm_wide.hip")
    # with [K, N] weights (3 kernels) 16 transposing reads for the first half of a step and 32 in each of its
    # four copies; two scales for either tile height in the scaled ones (2)
    assert build.check_gemm_waits(path) == 3 * (16 + 4 * 32) + 2 * 4
