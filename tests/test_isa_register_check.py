"""The build checks the compiler's assembly of every kernel for registers that are read and never written
(nnlib.jl_amd/csrc/check_isa_registers.py; the Makefile runs it on each object).  These cases pin the checker itself on
hand-written fragments: the miscompile it exists for (a matrix operand a[156:159] of which only a[156:158] is
reloaded), destinations it must recognise (loads, cross-lane reads, matrix results), and the registers the hardware
initialises."""
import importlib.util
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
spec = importlib.util.spec_from_file_location("check_isa_registers", os.path.join(ROOT, "nnlib.jl_amd", "csrc", "check_isa_registers.py"))
chk = importlib.util.module_from_spec(spec)
spec.loader.exec_module(chk)

HEAD = "\t.text\n\t.globl\tkern\nkern:\n"
TAIL = "\ts_endpgm\n\t.section\t.rodata,\"a\",@progbits\n\t.amdhsa_kernel kern\n\t.end_amdhsa_kernel\n"


def run(tmp_path, body):
    f = tmp_path / "k.s"
    f.write_text(HEAD + body + TAIL)
    return chk.check(str(f))


def test_partial_reload_is_found(tmp_path):
    body = ("\tds_read_b128 v[10:13], v0\n"
            "\tv_accvgpr_write_b32 a171, v13           ;  Reload Reuse\n"
            "\tscratch_load_dwordx3 a[156:158], off, off ; 12-byte Folded Reload\n"
            "\tv_accvgpr_write_b32 a56, v1\n"
            "\tv_mfma_f32_32x32x16_bf16 a[56:71], v[10:13], a[156:159], a[56:71]\n"
            "\tv_accvgpr_read_b32 v20, a60\n"
            "\tglobal_store_dword v[10:11], v20, off\n")
    found = run(tmp_path, body)
    assert any("a159" in f for f in found), found
    # a57 .. a71 are never written before the matrix instruction reads them as its accumulator input either
    assert all(("a159" in f) or any(f"a{i} " in f for i in range(57, 72)) for f in found), found


def test_clean_kernel_passes(tmp_path):
    body = ("\tv_lshlrev_b32_e32 v3, 2, v0\n"                       # v0: work-item id, set by the hardware
            "\tds_read_b128 v[10:13], v3\n"
            "\tds_read_b64_tr_b16 v[14:15], v3 offset:64\n"
            "\tds_bpermute_b32 v16, v3, v10\n"
            "\tscratch_load_dwordx4 a[0:3], off, off\n"
            "\tv_accvgpr_mov_b32 a4, a0\n"
            "\tv_mov_b32_e32 v17, 0\n"
            "\tv_mov_b32_e32 v18, 0\n"
            "\tv_mov_b32_e32 v19, 0\n"
            "\tv_mov_b32_e32 v20, 0\n"
            "\tv_mfma_f32_16x16x32_bf16 v[17:20], v[10:13], a[0:3], v[17:20]\n"
            "\tv_add_f32_e32 v21, v16, v14\n"
            "\tv_add_f32_e32 v21, v21, v15\n"
            "\tv_accvgpr_read_b32 v22, a4\n"
            "\tglobal_store_dwordx4 v[10:11], v[17:20], off\n"
            "\tglobal_store_dwordx2 v[10:11], v[21:22], off\n")
    assert run(tmp_path, body) == []


def test_two_kernels_are_checked_apart(tmp_path):
    f = tmp_path / "two.s"
    f.write_text(HEAD + "\tv_mov_b32_e32 v5, 1\n\tglobal_store_dword v[0:1], v5, off\n" + TAIL
                 + "\t.globl\tother\nother:\n\tglobal_store_dword v[0:1], v5, off\n\ts_endpgm\n\t.amdhsa_kernel other\n\t.end_amdhsa_kernel\n")
    found = chk.check(str(f))
    assert len(found) == 1 and "other" in found[0] and "v5" in found[0], found


def test_scratch_of_kernels_that_have_none(tmp_path):
    """A 128-wide Float32 kernel that spills is found, and a 64-wide one with bias / mask code (one took 588 bytes a lane once,
    for the code of a dropout that its calls did not have; another 20 with the dropout that they had); the 64-wide ones without
    that code may."""
    def described(name, scratch):
        return f"\t.amdhsa_kernel {name}\n\t\t.amdhsa_private_segment_fixed_size {scratch}\n\t.end_amdhsa_kernel\n"
    kern = "_ZN12_GLOBAL__N_114flash32_kernelILi%dELi1ELb1ELb%dELb0ELb1EEEv9FlashArgs"
    for file in ("attention_flash32-hip-amdgcn.s", "attention_flash32_drop-hip-amdgcn.s"):
        f = tmp_path / file
        for head, extras in ((128, 1), (128, 0), (64, 1)):
            f.write_text(described(kern % (head, extras), 588) + described(kern % (64, 0), 28))
            found = chk.check(str(f))
            assert len(found) == 1 and kern % (head, extras) in found[0] and "588" in found[0], found
            f.write_text(described(kern % (head, extras), 0))
            assert chk.check(str(f)) == []
    g = tmp_path / "attention_flash16_bf16_d64-hip-amdgcn.s"
    g.write_text(described("_ZN12_GLOBAL__N_114flash16_kernelILi1ELb0ELi0ELb0EfLb0EEEv9FlashArgs", 4)
                 + described("_ZN12_GLOBAL__N_114flash16_kernelILi1ELb0ELi7ELb0EfLb1EEEv9FlashArgs", 12))
    assert len(chk.check(str(g))) == 1
    h = tmp_path / "attention_backward_pair16_bf16-hip-amdgcn.s"
    for scratch, findings in ((12, 0), (152, 1)):   # as it was with bias entries loaded on both sides of the causal test
        h.write_text(described("_ZN12_GLOBAL__N_115bwd_pair_kernelILb1ELi5ELi0ELi2ELi8EEEv9FlashArgs13AttnBwdParams", scratch))
        assert len(chk.check(str(h))) == findings
