"""Build-level checks of the hand-written kernels that need no GPU.

The four-wave GEMM issues its v_mfma_f32_16x16x32 instructions as assembly
statements with the accumulator tied to the result (zdraw_amd/csrc/gemm_half.hip,
mfma16). The compiler adds no wait states around assembly, so anything it places
on its own between such an MFMA and the `s_nop 15` that ends the run (a copy or a
spill of an accumulator) would read the register before the MFMA has written it.
The check compiles the file to gfx950 assembly and fails on any such instruction.
"""
import os
import re
import shutil

import pytest

from zdraw_amd import build


@pytest.mark.skipif(not (os.path.exists("/opt/rocm/bin/hipcc") or shutil.which("hipcc")), reason="needs hipcc")
def test_nothing_reads_an_accumulator_inside_a_run_of_tied_mfmas():
    bad = build.tied_mfma_hazards()
    assert not bad, "\n".join(bad[:20])


@pytest.mark.skipif(not (os.path.exists("/opt/rocm/bin/hipcc") or shutil.which("hipcc")), reason="needs hipcc")
def test_only_the_source_writes_m0_in_the_four_wave_gemm():
    # its slab loads come in runs of four that share one M0 (attn_device.hpp, lds_dma_base): the
    # compiler does not know M0 is live between them, so it must not have put a write of its own there
    bad = build.m0_writes()
    assert not bad, "\n".join(bad[:20])


@pytest.mark.skipif(not (os.path.exists("/opt/rocm/bin/hipcc") or shutil.which("hipcc")), reason="needs hipcc")
def test_wide_head_kernel_keeps_its_accumulators_in_place_and_its_loop_free_of_spills():
    # attn_wide.hip: every MFMA of attn_wide_kernel is an assembly statement with the accumulator
    # tied to the result; nothing else may touch the accumulation file before the wait that ends a
    # step, and the blocks that hold the MFMAs may not use scratch memory
    bad = build.wide_mfma_hazards()
    assert not bad, "\n".join(bad[:20])


@pytest.mark.skipif(not (os.path.exists("/opt/rocm/bin/hipcc") or shutil.which("hipcc")), reason="needs hipcc")
def test_wide_head_kernel_leaves_m0_alone_and_no_load_reads_a_scalar_register_too_early():
    # its blocks come in runs of four loads that share one M0; and the compiler knows of no load in the
    # assembly statements, so it keeps no distance between them and a scalar register it restores
    src = os.path.join(build.CSRC, "attn_wide.hip")
    bad = build.m0_writes(src, "attn_wide_kernel") + build.vmem_sgpr_hazards(src) + build.vmem_sgpr_hazards(os.path.join(build.CSRC, "gemm_half.hip"))
    assert not bad, "\n".join(bad[:20])


@pytest.mark.skipif(not (os.path.exists("/opt/rocm/bin/hipcc") or shutil.which("hipcc")), reason="needs hipcc")
@pytest.mark.parametrize("name", ["attn_fwd.hip", "attn_wide.hip", "gemm_half.hip", "qk_prepass.hip"])
def test_no_kernel_reads_past_its_arguments(name):
    # the head of the pre-pass loads a word of each of its arguments' cache lines through the argument pointer
    # (qk_prepass.hip, touch_args): all of them have to lie within the segment that the kernel is launched with
    bad = build.kernarg_overreads(os.path.join(build.CSRC, name))
    assert not bad, "\n".join(bad[:20])


@pytest.mark.parametrize("load,over", [("s_load_dword s6, s[0:1], 0x3c", False), ("s_load_dword s6, s[0:1], 0x40", True),
                                       ("s_load_dwordx4 s[8:11], s[0:1], 0x30", False), ("s_load_dwordx4 s[8:11], s[0:1], 0x34", True),
                                       ("s_mov_b64 s[4:5], s[0:1]\n\ts_cmp_lg_u32 s4, 0\n\ts_load_dword s6, s[4:5], 0x40", True),
                                       ("s_load_dwordx2 s[0:1], s[0:1], 0x38\n\ts_load_dword s6, s[0:1], 0x40", False)])
def test_the_check_of_reads_past_the_arguments_sees_them(monkeypatch, load, over):
    asm = f"kern:\n; %bb.0:\n\t{load}\n\ts_endpgm\n\t.amdhsa_kernel kern\n\t\t.amdhsa_kernarg_size 64\n\t\t.amdhsa_user_sgpr_dispatch_ptr 0\n\t.end_amdhsa_kernel"
    monkeypatch.setattr(build, "_device_asm", lambda *_: asm.split("\n"))
    assert bool(build.kernarg_overreads("")) == over


@pytest.mark.skipif(not (os.path.exists("/opt/rocm/bin/hipcc") or shutil.which("hipcc")), reason="needs hipcc")
@pytest.mark.parametrize("name", ["attn_fwd.hip", "attn_wide.hip", "gemm_half.hip"])
def test_no_result_of_an_assembly_mfma_is_used_early(name):
    # attn_wide.hip forms its scores in ordinary registers with assembly MFMAs: what reads them has to
    # stand as far behind as the compiler would have put it
    bad = build.early_mfma_result_uses(os.path.join(build.CSRC, name))
    assert not bad, "\n".join(bad[:20])


M = "v_mfma_f32_16x16x32_bf16 v[4:7], v[8:11], v[12:15], "


@pytest.mark.parametrize("asm,early", [
    (["!" + M + "v[4:7]", "s_nop 6", "v_max_f32_e32 v0, v5, v5"], True),
    (["!" + M + "v[4:7]", "s_nop 7", "v_max_f32_e32 v0, v5, v5"], False),
    (["!" + M + "v[4:7]", "s_nop 6", "v_mov_b32_e32 v7, 0"], True),  # written over
    (["!" + M + "v[4:7]", "s_nop 6", "scratch_store_dwordx4 off, v[4:7], off"], True),  # spilled
    (["!" + M + "0", "v_add_f32_e32 v0, v1, v2", "!" + M + "v[4:7]", "s_nop 6", "v_exp_f32_e32 v0, v4"], True),  # the chain's last counts
    (["!" + M + "0", "!" + M + "v[4:7]", "s_nop 7", "v_exp_f32_e32 v0, v4"], False),
    (["!" + M + "0", ".LBB0_1:", "s_nop 7", "v_exp_f32_e32 v0, v4"], True),  # others may come in here
    ([M + "0", "v_exp_f32_e32 v0, v4"], False),  # the compiler's own
    (["!" + M.replace("v[4:7]", "a[4:7]") + "a[4:7]", "v_exp_f32_e32 v0, v4"], False),
])
def test_the_check_of_early_uses_sees_them(monkeypatch, asm, early):
    lines = ["kern:"]
    for a in asm:
        lines += [";;#ASMSTART", "\t" + a[1:], ";;#ASMEND"] if a.startswith("!") else ["\t" + a]
    monkeypatch.setattr(build, "_device_asm", lambda *_: lines)
    assert bool(build.early_mfma_result_uses("")) == early


@pytest.mark.skipif(not (os.path.exists("/opt/rocm/bin/hipcc") or shutil.which("hipcc")), reason="needs hipcc")
def test_no_load_of_the_attention_kernel_reads_a_scalar_register_too_early():
    bad = build.vmem_sgpr_hazards(os.path.join(build.CSRC, "attn_fwd.hip"))
    assert not bad, "\n".join(bad[:20])


LOAD = "buffer_load_dwordx4 v4, s[8:11], s5 offen lds"


@pytest.mark.parametrize("asm,early", [
    (["v_readfirstlane_b32 s5, v1", LOAD], True),
    (["v_readfirstlane_b32 s5, v1", "s_cmp_lg_u32 s5, 0", LOAD], True),  # only reads it
    (["v_readfirstlane_b32 s5, v1", "s_bitcmp1_b32 s5, 0", LOAD], True),
    (["v_readfirstlane_b32 s5, v1", "s_nop 3", LOAD], True),
    (["v_readfirstlane_b32 s5, v1", "s_nop 4", LOAD], False),
    (["v_readfirstlane_b32 s5, v1", "s_cmp_lg_u32 s5, 0", "s_nop 3", LOAD], False),
    (["v_readfirstlane_b32 s5, v1", "s_mov_b32 s5, s6", LOAD], False),  # written over
    (["v_readfirstlane_b32 s5, v1", "s_mov_b64 s[4:5], s[6:7]", LOAD], False),
    (["v_readfirstlane_b32 s5, v1", "s_add_u32 s6, s5, 4", LOAD], True),
    (["v_readlane_b32 s10, v255, 3", LOAD], True),  # the descriptor
    (["v_cmp_gt_i32_e64 s[4:5], s6, v0", LOAD], True),
    (["v_readfirstlane_b32 s6, v1", LOAD], False),
])
def test_the_check_of_scalar_registers_sees_early_reads(monkeypatch, asm, early):
    monkeypatch.setattr(build, "_device_asm", lambda *_: ["kern:"] + asm)
    assert bool(build.vmem_sgpr_hazards("")) == early


@pytest.mark.skipif(not (os.path.exists("/opt/rocm/bin/hipcc") or shutil.which("hipcc")), reason="needs hipcc")
@pytest.mark.parametrize("name", ["attn_fwd.hip", "attn_wide.hip", "gemm_half.hip", "qk_prepass.hip"])
def test_nothing_writes_the_data_of_a_store_right_behind_it(name):
    # attn_device.hpp, store_through: the compiler knows of no store in an assembly statement
    bad = build.early_store_data_writes(os.path.join(build.CSRC, name))
    assert not bad, "\n".join(bad[:20])


STORE = "global_store_dwordx4 v[2:3], v[4:7], off sc1"


@pytest.mark.parametrize("asm,early", [
    ([STORE, "v_add_u32_e32 v4, 1, v0"], True),
    ([STORE, "s_nop 0", "v_add_u32_e32 v7, 1, v0"], True),
    ([STORE, "s_nop 1", "v_add_u32_e32 v7, 1, v0"], False),
    ([STORE, "s_add_u32 s0, s0, 1", "v_pk_mul_f16 v5, v0, v1"], True),
    ([STORE, "s_nop 0", "v_add_u32_e32 v2, 1, v4"], False),  # the address, and reads
    ([STORE, "s_nop 0", ".LBB0_1:", "v_mov_b64_e32 v[6:7], v[0:1]"], True),
    ([STORE, "v_permlane32_swap_b32_e32 v0, v6"], True),
    (["buffer_store_dwordx4 v[4:7], v2, s[0:3], 0 offen", "v_mov_b32_e32 v4, 0"], True),
    (["global_store_dwordx2 v[2:3], v[4:5], off sc1", "v_mov_b32_e32 v4, 0"], False),
])
def test_the_check_of_store_data_sees_early_writes(monkeypatch, asm, early):
    monkeypatch.setattr(build, "_device_asm", lambda *_: ["kern:"] + asm)
    assert bool(build.early_store_data_writes("")) == early


@pytest.mark.skipif(not (os.path.exists("/opt/rocm/bin/hipcc") or shutil.which("hipcc")), reason="needs hipcc")
def test_which_products_store_their_rows_through_the_l2():
    # gemm_half.hip, store_rows_lds: tiles of 128 x 96 on, but not 16-bit C of a ragged k, whose rows begin
    # anywhere in a cache line
    kernel, seen = None, {}
    for line in build._device_asm(os.path.join(build.CSRC, "gemm_half.hip")):
        text = line.split(";")[0].strip()
        name = re.match(r"^_ZN\w*gemm_pipe_kernelILb[01]E([ft])Li(\d)ELi(\d)ELi\d+ELb([01])E\w*:$", text)
        if name or (text.endswith(":") and not text.startswith(".")):
            kernel = text if name else None
            if name:
                seen[kernel] = (name.groups(), set())
        elif kernel and text.startswith("global_store_dwordx4"):
            seen[kernel][1].add("sc1" in text.split())
    assert len(seen) == 72
    for (c, ti, tj, ragged), through in seen.values():
        assert through == {int(ti) * int(tj) >= 12 and (c == "f" or ragged == "0")}, (c, ti, tj, ragged)


@pytest.mark.skipif(not (os.path.exists("/opt/rocm/bin/hipcc") or shutil.which("hipcc")), reason="needs hipcc")
def test_which_builds_form_the_lanes_number_again_for_the_key_block_list():
    # attn_fwd.hip, list_load: of the masked builds that norm K in the tile load (eight waves) only those of bf16 rows
    # with a bound; the others lose 1 to 14 % by it. (All form it in their steps' mask branches.)
    kernel, seen = None, {}
    for line in build._device_asm(os.path.join(build.CSRC, "attn_fwd.hip")):
        text = line.split(";")[0].strip()
        name = re.match(r"^_ZN\w*attn_fwd_kernelI(f|DF16b)Li([12])ELb1ELb([01])ELi1ELi8ELb0ELi1E\w*:$", text)
        if name or (text.endswith(":") and not text.startswith(".")):
            kernel = name.groups() if name else None
            if name:
                seen[kernel] = 0
        elif kernel and text.startswith("v_mbcnt_lo"):
            seen[kernel] += 1
    assert len(seen) == 8
    fewest = min(seen.values())
    for (rows, _, bounded), n in seen.items():
        assert (n > fewest) == (rows == "DF16b" and bounded == "1"), seen
