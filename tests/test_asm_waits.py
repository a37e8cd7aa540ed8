"""The check of hand-counted waits (moonep_amd/asm_waits.py): on pieces of assembly that are right and
wrong in one place each, and on what the compiler makes of the GEMM kernels."""

import pytest

from moonep_amd import asm_waits, build

LDS = "ds_read_b64_tr_b16 v[4:5], v9 offset:0"
VMEM = "global_load_dword v4, v[2:3], off"


def _kernel(*lines, spills=0):
    body = "\n".join(l if l.endswith(":") else f"\t{l}" for l in lines)
    return (f"gemm_k:                                 ; @gemm_k\n{body}\n\ts_endpgm\n.Lfunc_end0:\n"
            f"amdhsa.kernels:\n  - .agpr_count: 0\n    .name:           gemm_k\n    .vgpr_spill_count: {spills}\n")


def _asm(text):
    return (";;#ASMSTART", text, ";;#ASMEND")


LOOP = (*_asm(VMEM), ".LBB0_1:", "buffer_load_dwordx4 v8, s[0:3], 0 offen lds", "s_waitcnt vmcnt(2)", "s_cbranch_scc1 .LBB0_1")


@pytest.mark.parametrize("lines", [
    (*_asm(LDS), "v_add_u32 v6, v7, v8", "s_waitcnt vmcnt(3) lgkmcnt(0)", *_asm("; arrived v[4:5]"), "v_mov_b32 v1, v4"),
    (*_asm(VMEM), "global_load_dword v8, v[2:3], off", "s_waitcnt vmcnt(1)", *_asm("; arrived v4"), "v_mov_b32 v1, v4"),
    # covered on the way round or behind the loop
    (*LOOP, "s_waitcnt vmcnt(1)", *_asm("; arrived v4")),
    (*_asm(LDS), "s_cbranch_vccz .LBB0_2", "s_waitcnt lgkmcnt(0)", "v_mov_b32 v4, 0", ".LBB0_2:", "s_waitcnt lgkmcnt(0)",
     *_asm("; arrived v[4:5]")),
])
def test_right(lines):
    assert asm_waits.check(_kernel(*lines)) == ([], 1)


@pytest.mark.parametrize("lines", [
    (*_asm(LDS), "v_mov_b32 v1, v5", "s_waitcnt lgkmcnt(0)", *_asm("; arrived v[4:5]")),        # read
    (*_asm(LDS), "v_pk_mul_f16 v[3:4], v[6:7], v8", "s_waitcnt lgkmcnt(0)"),                    # overwritten
    (*_asm(LDS), "s_waitcnt lgkmcnt(1)", *_asm("; arrived v[4:5]")),                            # not waited for
    (*_asm(LDS), "s_waitcnt vmcnt(0)", *_asm("; arrived v[4:5]")),                              # another counter
    (*_asm(VMEM), "s_waitcnt vmcnt(1)", *_asm("; arrived v4")),                                 # nothing younger
    (*_asm(VMEM), "global_store_dword v[2:3], v8, off", "s_waitcnt vmcnt(1)", *_asm("; arrived v4")),
    (*LOOP, *_asm("; arrived v4")),                                                             # one round covers too little
    (*_asm(LDS), "s_cbranch_vccz .LBB0_2", "s_waitcnt lgkmcnt(0)", ".LBB0_2:", *_asm("; arrived v[4:5]")),
    (*_asm(VMEM), ".LBB0_1:", "v_mov_b32 v1, v4", "s_waitcnt vmcnt(0)", "s_branch .LBB0_1"),
])
def test_wrong(lines):
    faults, followed = asm_waits.check(_kernel(*lines))
    assert followed == 1 and len(faults) == 1 and "line" in faults[0]


def test_a_spill_is_a_fault_and_a_path_that_cannot_be_followed_an_error():
    right = (*_asm(LDS), "s_waitcnt lgkmcnt(0)", *_asm("; arrived v[4:5]"))
    assert "vgpr_spill_count 2" in asm_waits.check(_kernel(*right, spills=2))[0][0]
    with pytest.raises(ValueError, match="cannot be followed"):
        asm_waits.check(_kernel(*_asm(LDS), "s_setpc_b64 s[0:1]"))


def test_the_gemm_kernels_as_they_are_compiled(tmp_path):
    path = str(tmp_path / "gemm.s")
    build.gemm_assembly(path)
    # 16 transposing reads in each kernel with [K, N] weights (3), 48 in the weight gradient, two
    # scales in each of the scaled (2); 8 for every unit of a streaming tile of 1 to 4, alone and in pairs
    assert build.check_gemm_waits(path) == 3 * 16 + 48 + 2 * 2 + 2 * 8 * (1 + 2 + 3 + 4)
