"""The build's reading of kernels that keep sums in named accumulation registers (check_acc.py), on assembly written here."""
import importlib.util
import os

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llm_metal_amd", "csrc")
spec = importlib.util.spec_from_file_location("check_acc", os.path.join(CSRC, "check_acc.py"))
check_acc = importlib.util.module_from_spec(spec)
spec.loader.exec_module(check_acc)

KERNEL = """
k_sums:                                 ; @k_sums
; %bb.0:
	ds_read_b128 v[0:3], v20
	{ahead}
	s_waitcnt lgkmcnt(0)
	{near}
	;;#ASMSTART
	v_mfma_f32_16x16x32_f16 a[4:7], v[0:3], v[8:11], a[4:7]
	;;#ASMEND
	{behind}
	;;#ASMSTART
	v_accvgpr_read_b32 v12, a4
	;;#ASMEND
	s_endpgm
	.section	.rodata
	.amdhsa_kernel k_sums
		.amdhsa_private_segment_fixed_size {scratch}
	.end_amdhsa_kernel
k_other:                                ; @k_other
	v_accvgpr_write_b32 a0, v1          ; (a kernel that leaves its accumulators to the compiler)
	v_mfma_f32_32x32x16_f16 a[0:15], v[0:3], v[8:11], a[0:15]
	s_endpgm
"""


def kernel(**kw):
    return KERNEL.format(**{"ahead": "v_add_u32_e32 v30, v0, v1", "near": "s_nop 0", "behind": "v_mov_b32_e32 v8, v9", "scratch": 0, **kw})


def test_a_sound_kernel_passes():
    assert check_acc.faults(kernel()) == ([], 1)
    assert check_acc.faults(kernel(ahead="v_mov_b32_e32 v8, v9", near="s_nop 1"))[0] == []          # two wait states between
    assert check_acc.faults(KERNEL.split("k_other")[1])[1] == 0


@pytest.mark.parametrize("kw", [dict(behind="v_accvgpr_write_b32 a9, v1"), dict(behind="global_load_dwordx4 a[16:19], v[2:3], off"), dict(ahead="v_accvgpr_mov_b32 a200, a4"),
                                dict(scratch=16), dict(behind="scratch_store_dword off, v1, off"), dict(behind="s_swappc_b64 s[30:31], s[4:5]"),
                                dict(near="v_mov_b32_e32 v9, v40"), dict(near="v_mov_b64_e32 v[2:3], v[40:41]"), dict(ahead="v_mov_b32_e32 v9, v40", near="")],
                         ids=["write", "load", "move", "scratch", "spill", "call", "operand", "operand_pair", "operand_two_ahead"])
def test_an_unsound_kernel_is_refused(kw):
    found, kernels = check_acc.faults(kernel(**kw))
    assert kernels == 1 and len(found) == 1, found


def test_files_without_such_a_kernel_are_refused(tmp_path, capsys):
    f = tmp_path / "x.s"
    f.write_text("k:\n\ts_endpgm\n")
    assert check_acc.main([str(f)]) and "no kernel" in capsys.readouterr().err
    f.write_text(kernel())
    assert not check_acc.main([str(f)])
