"""The build-time checks of the generated code (relax_amd/check_ring_asm.py), on small
hand-written listings: what they must accept and what they must refuse."""
from relax_amd import check_ring_asm as c

KERNEL = """
_ZN2wq4testEv:
\ts_load_dwordx2 s[0:1], s[4:5], 0x0
\t;;#ASMSTART
\tglobal_load_dwordx4 v[2:5], v6, s[0:1] nt
\t;;#ASMEND
{body}
\ts_endpgm
.Lfunc_end0:
"""


def _errors(body):
    return c.check(KERNEL.format(body=body))


def test_ring_registers_may_only_be_read_by_the_unpack_instructions():
    ok = "\t;;#ASMSTART\n\ts_waitcnt vmcnt(0)\n\t;;#ASMEND\n\t;;#ASMSTART\n\tv_and_or_b32 v7, v2, s2, v8\n\t;;#ASMEND\n\tv_add_u32_e32 v9, v7, v7"
    assert _errors(ok) == []
    assert _errors("\tv_mov_b32_e32 v9, v3") and "v_mov_b32_e32" in _errors("\tv_mov_b32_e32 v9, v3")[0]      # a copy
    assert _errors("\tscratch_store_dwordx4 off, v[2:5], off offset:16")                                            # a spill
    assert _errors("\tv_lshrrev_b32_e32 v9, 4, v2")                                                                 # another shift
    assert _errors("\tv_mov_b32_dpp v9, v2 quad_perm:[0,1,2,3] row_mask:0xf bank_mask:0xf") == []                   # the lane exchange
    # a register the compiler reuses as a temporary after the slot was consumed is no longer a ring register
    assert _errors("\tv_mov_b32_e32 v2, 0\n\tv_add_u32_e32 v9, v2, v2") == []


def test_a_kernel_with_a_ring_must_not_spill_any_register():
    spill = "\tscratch_store_dword off, v40, off offset:84\n\tscratch_load_dword v40, off, off offset:84"
    errs = _errors(spill)
    assert errs and "scratch accesses" in errs[0]
    assert _errors("\tv_add_u32_e32 v40, v41, v42") == []


def test_a_file_without_ring_loads_is_refused():
    assert c.check("_ZN2wq4testEv:\n\tv_mov_b32_e32 v0, 0\n\ts_endpgm\n.Lfunc_end0:\n")


def _hazards(body):
    return c.check_asm_results(KERNEL.format(body=body))


def test_inline_assembly_results_must_not_reach_mfma_or_dpp_at_once():
    asm = "\t;;#ASMSTART\n\tv_pk_mul_f16 v10, v11, v12 op_sel_hi:[1,0]\n\t;;#ASMEND\n"
    mfma = "\tv_mfma_f32_16x16x32_f16 v[20:23], v[10:13], v[30:33], v[20:23]\n"
    filler = "\tv_add_u32_e32 v40, v41, v42\n"
    assert _hazards(asm + mfma)                                   # directly behind
    assert _hazards(asm + filler + mfma)                          # one instruction between
    assert _hazards(asm + filler + filler + filler + mfma) == []  # far enough
    assert _hazards("\tv_pk_mul_f16 v10, v11, v12\n" + mfma) == []  # the compiler's own instruction: its business
    # a statement that ends in its own s_nop is safe wherever it is placed
    own = "\t;;#ASMSTART\n\tv_mov_b32_dpp v10, v2 quad_perm:[0,1,2,3] row_mask:0xf bank_mask:0xf\n\ts_nop 1\n\t;;#ASMEND\n"
    dpp = "\tv_mov_b32_dpp v50, v10 row_ror:8 row_mask:0xf bank_mask:0xc\n"
    assert _hazards(own + dpp) == []
    bare = "\t;;#ASMSTART\n\tv_mov_b32_dpp v10, v2 quad_perm:[0,1,2,3] row_mask:0xf bank_mask:0xf\n\t;;#ASMEND\n"
    assert _hazards(bare + dpp)
    assert _hazards(bare + "\tv_mov_b32_dpp v10, v51 row_ror:8 row_mask:0xf bank_mask:0xc\n")  # the old value of a DPP destination counts
    # loads inside inline assembly are waited for by s_waitcnt, not by wait states
    assert _hazards("\t;;#ASMSTART\n\tglobal_load_dwordx4 v[10:13], v6, s[0:1] nt\n\t;;#ASMEND\n" + mfma) == []


GEMM = """
_ZN2wq15gemm_lds_kernelEv:
\tbuffer_load_dwordx4 v1, s[0:3], 0 offen lds
.LBB0_1:
\ts_waitcnt vmcnt(3) lgkmcnt(0)
\ts_barrier
\tbuffer_load_dwordx4 v1, s[0:3], s4 offen lds
\ts_cbranch_scc1 .LBB0_1
{tail}
\ts_endpgm
.Lfunc_end0:
"""


def test_direct_loads_have_landed_in_front_of_the_staging():
    def errors(tail, text=GEMM):
        return c.check_direct_loads_drained(text.format(tail=tail))

    wait, barrier, write = "\ts_waitcnt vmcnt(0)\n", "\ts_barrier\n", "\tds_write_b128 v2, v[4:7]"
    assert errors(wait + barrier + write) == []
    assert errors("\ts_waitcnt vmcnt(0) lgkmcnt(0)\n" + barrier + write) == []
    assert errors(write)                                        # the loop ends with loads on their way
    assert errors(barrier + write)
    assert errors(barrier + wait + write)                       # the barrier lies in front of the wait
    assert "other wavefronts" in errors(wait + write)[0]        # those of the others may still be
    assert errors("\ts_waitcnt vmcnt(1)\n" + barrier + write)
    # one way around the wait is enough
    assert errors("\ts_cbranch_vccz .LBB0_3\n" + wait + barrier + ".LBB0_3:\n" + write)
    # a second tile body behind the first
    again = "\tglobal_load_lds_dwordx4 v[2:3], off\n"
    assert errors(wait + barrier + write + "\n" + again + write)
    assert errors(wait + barrier + write + "\n" + again + wait + barrier + write) == []
    # nothing to check, or other kernels only
    assert errors(write, GEMM.replace(" lds", ""))
    assert errors(write, GEMM.replace("gemm_lds", "other"))


def test_loads_past_the_end_have_no_scalar_offset():
    def errors(body, text=GEMM):
        return c.check_empty_descriptors(text.replace("s4 offen", "s9 offen").format(tail="").replace(".LBB0_1:\n", body + ".LBB0_1:\n"))

    assert errors("\ts_cselect_b32 s9, s20, 0\n") == []
    assert errors("\ts_cselect_b32 s9, 0, 0x80\n") == []
    assert errors("\ts_and_b32 s9, s20, s2\n") == []
    assert errors("\ts_cselect_b32 s8, s20, 0\n\ts_mov_b32 s9, s8\n") == []
    assert errors("\ts_mov_b32 s9, 0\n") == []
    assert errors("")                                                     # written nowhere
    assert errors("\ts_lshl_b32 s9, s20, 7\n")
    assert errors("\ts_cselect_b32 s9, s20, s21\n")
    assert errors("\ts_mov_b32 s9, s20\n")
    assert errors("\ts_cselect_b32 s9, s20, 0\n\ts_add_i32 s9, s9, 64\n")  # written again
    assert errors("\ts_cselect_b32 s9, s20, 0\n\ts_mul_hi_u32 s9, s1, s2\n")
    assert errors("\ts_cselect_b32 s9, s20, 0\n\ts_lshl_b64 s[8:9], s[20:21], 1\n")
    # on one of two ways only
    assert errors("\ts_cbranch_vccz .LBB0_1\n\ts_cselect_b32 s9, s20, 0\n")
    # behind the load, so not in the second round of the loop
    late = GEMM.replace("s4 offen", "s9 offen").replace("\ts_cbranch", "\ts_add_i32 s9, s9, 128\n\ts_cbranch")
    assert errors("\ts_cselect_b32 s9, s20, 0\n", late)
    assert errors("\ts_cselect_b32 s9, s20, 0\n", GEMM.replace("gemm_lds", "other"))


LIST = """
_ZN2wq{kernel}ILb0ELi2EEEvPKNS_12GemvListDescE:
{body}
\tbuffer_load_dwordx4 v[2:5], v6, s[12:15], s9 offen
\ts_endpgm
.Lfunc_end0:
"""


def test_loads_of_the_lists_of_several_rows_past_the_end_have_no_scalar_offset(monkeypatch):
    import pytest

    source = "q4g32_batch_list.hip"
    assert c.GUARDED_KERNELS[source]
    for kernel in c.GUARDED_KERNELS[source]:
        bad, good = (LIST.format(kernel=kernel, body=b) for b in ("\ts_lshl_b32 s9, s20, 4", "\ts_and_b32 s9, s20, s21"))
        assert c.check_empty_descriptors(bad, kernel) and c.check_empty_descriptors(good, kernel) == []
        with_others = "".join(LIST.format(kernel=k, body="\ts_mov_b32 s9, 0") for k in c.GUARDED_KERNELS[source] if k != kernel)
        monkeypatch.setattr(c, "check", lambda text: [])
        monkeypatch.setattr(c, "_assembly", lambda *a: bad + with_others)
        with pytest.raises(RuntimeError, match="past the end"):
            c.check_source("hipcc", [], source)
        monkeypatch.setattr(c, "_assembly", lambda *a: good + with_others)
        c.check_source("hipcc", [], source)


def test_the_build_checks_every_source_with_the_tiled_gemm():
    import os

    csrc = os.path.join(c.HERE, "csrc")
    with_gemm = set()
    for name in os.listdir(csrc):
        if name.endswith(".hip"):
            with open(os.path.join(csrc, name)) as f:
                if "launch_gemm_lds<" in f.read():
                    with_gemm.add(name)
    assert with_gemm == set(c.DIRECT_LOAD_SOURCES)


HELD = """
_ZN2wq16held_gemm_kernelEv:
\t;;#ASMSTART
\tv_mov_b32 v10, v2
{nop}\t;;#ASMEND
\tv_mov_b32_dpp v50, v10 row_ror:8 row_mask:0xf bank_mask:0xc
{body}
\ts_endpgm
.Lfunc_end0:
"""


def test_the_kernel_with_activations_in_registers_is_checked(monkeypatch):
    import os

    import pytest

    including = set()
    for name in os.listdir(os.path.join(c.HERE, "csrc")):
        if name.endswith(".hip"):
            with open(os.path.join(c.HERE, "csrc", name)) as f:
                if '#include "held_gemm.h"' in f.read():
                    including.add(name)
    assert including == set(c.HELD_SOURCES)
    monkeypatch.setattr(c, "check_direct_loads_drained", lambda text: [])
    monkeypatch.setattr(c, "check_empty_descriptors", lambda text: [])
    nop = "\ts_nop 1\n"
    for name in c.HELD_SOURCES:
        for text, refused in ((HELD.format(nop=nop, body=""), None), (HELD.format(nop="", body=""), "wait states"),
                              (HELD.format(nop=nop, body="\tscratch_store_dword off, v9, off offset:4"), "spilled"),
                              (HELD.format(nop=nop, body="").replace("held_gemm", "other"), "spilled")):
            monkeypatch.setattr(c, "_assembly", lambda *a, text=text: text)
            if refused is None:
                c.check_source("hipcc", [], name)
            else:
                with pytest.raises(RuntimeError, match=refused):
                    c.check_source("hipcc", [], name)


def test_an_incremental_build_does_not_keep_what_was_refused(tmp_path, monkeypatch):
    """A source that does not compile must not hide that another one was refused: its object would pass for up to date."""
    import os

    import pytest

    from relax_amd import build as b

    refused, broken, fine = "gptq.hip", "common.cc", "q4n32.hip"
    monkeypatch.setattr(b, "OBJDIR", str(tmp_path))
    monkeypatch.setattr(b, "sources", lambda: [os.path.join(b.CSRC, n) for n in (refused, broken, fine)])

    def compile_(src):
        if src.endswith(broken):
            raise RuntimeError("does not compile")
        (tmp_path / (os.path.basename(src) + ".o")).write_text("object")

    def check(name):
        if name == refused:
            raise RuntimeError("refused")

    monkeypatch.setattr(b, "_compile", compile_)
    monkeypatch.setattr(b, "check_asm", check)
    with pytest.raises(RuntimeError):
        b.build(verbose=False, incremental=True)
    assert sorted(p.name for p in tmp_path.iterdir()) == [fine + ".o"]
