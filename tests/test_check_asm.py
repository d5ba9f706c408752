"""The build's check of kernels with inline asm (csrc/check_asm.py), on short pieces of assembly (CPU only)."""
import importlib.util
import pathlib

import pytest

_PATH = pathlib.Path(__file__).resolve().parent.parent / "nano-vllm-triton-kernels_amd" / "csrc" / "check_asm.py"
_SPEC = importlib.util.spec_from_file_location("check_asm", _PATH)
check_asm = importlib.util.module_from_spec(_SPEC)
_SPEC.loader.exec_module(check_asm)

MFMA = "v_mfma_f32_32x32x16_bf16 v[0:15], v[16:19], a[0:3], v[0:15]"
ACC = "v_mfma_f32_32x32x16_bf16 a[16:31], v[20:23], v[24:27], a[16:31]"


def kernel(*code, scratch=0):
    lines = "\n".join("\t" + c if not c.endswith(":") else c for c in code)
    return (f"\t.type\tfoo_kernel,@function\nfoo_kernel: ; @foo_kernel\n{lines}\n\ts_endpgm\n\t.section .rodata\n"
            f"amdhsa.kernels:\n  - .agpr_count: 4\n    .name: foo_kernel\n    .private_segment_fixed_size: {scratch}\n")


@pytest.mark.parametrize("code,why", [
    ([MFMA, "s_nop 10", "v_add_f32_e32 v40, v15, v41"], "matrix result used"),
    ([MFMA, "s_nop 10", "v_mov_b32_e32 v3, 0"], "matrix result used"),
    ([ACC, ACC, "s_nop 10", "v_accvgpr_read_b32 v1, a31"], "matrix result used"),
    ([MFMA, "s_nop 7", "s_nop 2", "global_store_dwordx4 v[60:61], v[0:3], off"], "matrix result used"),
    ([MFMA, "v_mfma_f32_32x32x16_bf16 v[64:79], v[0:3], a[0:3], 0"], "another matrix instruction"),
    ([MFMA, "v_mfma_f32_32x32x16_bf16 v[8:23], v[30:33], a[0:3], v[8:23]"], "another matrix instruction"),
    (["v_mov_b32_e32 v17, v50", "s_add_i32 s0, s0, 1", MFMA], "read by a matrix instruction"),
    (["v_accvgpr_write_b32 a2, v50", MFMA], "read by a matrix instruction"),
    (["v_cvt_pk_bf16_f32 v25, v1, v2", ACC], "read by a matrix instruction"),
    ([".LBB0_1:", "v_cmp_gt_i32_e32 vcc, v50, v51", ACC, "s_nop 10", "s_cbranch_vccnz .LBB0_1", "s_branch .LBB0_2",
      ".LBB0_2:", "v_accvgpr_read_b32 v1, a16"], ""),   # 1 + 11 + 1 + 1 states on: fine
    ([".LBB0_1:", "v_accvgpr_read_b32 v1, a16", "s_nop 1", ACC, "s_cbranch_scc1 .LBB0_1"], "matrix result used"),
    (["v_readlane_b32 s4, v254, 3", "s_nop 3", "global_load_lds_dwordx4 v1, s[4:5]"], "scalar register"),
    (["v_readlane_b32 s4, v254, 3", "s_mov_b32 s4, 0", "global_load_lds_dwordx4 v1, s[4:5]"], ""),
    (["v_readfirstlane_b32 s4, v1", "s_nop 4", "buffer_load_dwordx4 v1, s[4:7], s8 offen lds"], ""),
    (["s_mov_b32 m0, s1", "buffer_load_dwordx4 v1, s[4:7], s8 offen lds"], "m0 written"),
    (["s_mov_b32 m0, s1", "s_nop 0", "buffer_load_dwordx4 v1, s[4:7], s8 offen lds"], ""),
    ([MFMA, MFMA, ACC, "s_nop 11", "v_add_f32_e32 v40, v15, v41"], ""),
    ([MFMA, "s_nop 11", "v_add_f32_e32 v40, v15, v41"], ""),
    ([MFMA, "v_add_f32_e32 v40, v42, v41", "ds_read_b128 v[16:19], v50"], ""),
    (["v_mov_b32_e32 v17, v50", "s_nop 1", MFMA], ""),
])
def test_distances(code, why):
    found = check_asm.check(kernel(*code), ["foo"])
    assert bool(found) == bool(why), found
    assert all(why in f for f in found)


def test_scratch_and_missing_kernels_are_reported():
    assert check_asm.check(kernel(MFMA), ["foo"]) == []
    assert "16 bytes of scratch" in check_asm.check(kernel(MFMA, scratch=16), ["foo"])[0]
    assert check_asm.check(kernel(MFMA), ["bar"]) == ["no kernel bar"]
