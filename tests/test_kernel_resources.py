"""Register and scratch use of the kernels that count their own vector-memory operations (CPU: hipcc compiles the
source to assembly for gfx950, nothing runs).

The sparse attention kernels issue their tile copies through inline asm and wait for them with
`s_waitcnt vmcnt(n)`, n being the number of operations issued since. A register spilled to scratch adds a
vector-memory operation that nobody counted, and its reload waits for every copy in flight. Zero scratch is
therefore part of these kernels' contract, not a tuning detail.

The second rule checked here: no inline asm statement loads into a register. The compiler takes an asm output for
valid as soon as the statement ends and may move, reuse or spill that register while the load is in flight; only
loads whose destination is LDS (they write no register) are issued through asm, every other load is an ordinary
one that the compiler waits for itself.
"""
import os
import shutil

import pytest

from moespresso_amd import build

pytestmark = pytest.mark.skipif(not (os.path.exists(build.HIPCC) or shutil.which(build.HIPCC)), reason="hipcc not installed")


@pytest.fixture(scope="module")
def sparse_assembly():
    return build.device_assembly(os.path.join(build.CSRC, "sparse_attn.hip"))


@pytest.fixture(scope="module")
def sparse_kernels(sparse_assembly):
    return build.kernel_resources(os.path.join(build.CSRC, "sparse_attn.hip"), sparse_assembly)


def test_sparse_attention_kernels_use_no_scratch(sparse_kernels):
    counted = {k: v for k, v in sparse_kernels.items() if "sparse_attn_split_kernel" in k or "sparse_attn_prefill_kernel" in k}
    # six instances of the split kernel (element type x row width x query type x rope) and the prefill consumer
    assert len(counted) == 7, sorted(counted)
    for name, res in counted.items():
        assert res["scratch_bytes"] == 0 and res["vgpr_spills"] == 0, (name, res)
        # eight waves per workgroup, one workgroup per CU: 256 registers per lane are there, not one more
        assert res["vgprs"] <= 256, (name, res)


def test_the_fp4_scores_with_the_float16_form_inside_fit_three_waves():
    """Three waves of a SIMD share 512 registers, in units of eight: 168 each, and nothing may be spilled to keep to that."""
    (name, res), = [(k, v) for k, v in build.kernel_resources(os.path.join(build.CSRC, "indexer_tiled.hip")).items() if "scores_fp4_kernel" in k]
    assert res["vgprs"] <= 168 and res["scratch_bytes"] == 0 and res["vgpr_spills"] == 0, (name, res)


def test_flash_prefill_spills_one_value_in_one_form_and_none_around_its_copies():
    """Float32 queries over an 8-bit prefix in fewer than four key ranges: one value is put away in front of the tile loops and
    fetched once behind the loop over 8-bit tiles, where the kernel has waited for all its copies."""
    source = os.path.join(build.CSRC, "flash_prefill.hip")
    text = build.device_assembly(source)
    bodies = build.kernel_bodies(text)
    spilling = {k for k, v in build.kernel_resources(source, text).items() if v["scratch_bytes"] or v["vgpr_spills"]}
    assert len(bodies) > 28 and all("flash_prefill_kernelILi1ELb1E" in k and "ELb1ELb1ELb0EEE" in k for k in spilling), sorted(spilling)
    for name in spilling:
        lines = [l.split(";")[0].strip() for l in bodies[name]]
        ops = [i for i, l in enumerate(lines) if l.startswith("scratch_")]
        first_tile = next(i for i, l in enumerate(lines) if l.startswith("v_mfma"))
        assert [lines[i].split()[0] for i in ops] == ["scratch_store_dword", "scratch_load_dword"], name
        assert ops[0] < first_tile < ops[1], name
        in_front = [l for l in lines[ops[1] - 6:ops[1]] if l and not l.startswith(".")]
        assert any(l.startswith("s_barrier") for l in in_front) and any("vmcnt(0)" in l for l in in_front), (name, in_front)


def test_resource_query_sees_every_kernel_of_the_source(sparse_kernels):
    assert sum("sparse_attn_merge_kernel" in k for k in sparse_kernels) == 3
    for res in sparse_kernels.values():
        assert set(res) == {"vgprs", "sgprs", "scratch_bytes", "vgpr_spills", "sgpr_spills"} and res["vgprs"] > 0


def test_no_inline_asm_statement_loads_into_a_register(sparse_assembly):
    bodies = build.kernel_bodies(sparse_assembly)
    assert any("sparse_attn_prefill_kernel" in k for k in bodies) and len(bodies) >= 11, sorted(bodies)
    for name, lines in bodies.items():
        assert build.inline_asm_register_loads(lines) == [], name
    # the rule has teeth: the same scan flags a register load inside an asm block
    sample = ["\t;;#ASMSTART", "\tglobal_load_dword v3, v[4:5], off", "\t;;#ASMEND",
              "\t;;#ASMSTART", "\tglobal_load_lds_dwordx4 v[4:5], off", "\t;;#ASMEND", "\tglobal_load_dword v9, v[4:5], off"]
    assert build.inline_asm_register_loads(sample) == ["global_load_dword v3, v[4:5], off"]


def test_prefill_consumer_store_count_matches_what_its_waits_assume(sparse_assembly):
    """The persistent prefill consumer counts sixteen output stores per unit and wave into its wait counts (a count
    above what was issued would end a wait early); the compiler must issue exactly that many, and no other store."""
    (name, lines), = [(k, v) for k, v in build.kernel_bodies(sparse_assembly).items() if "sparse_attn_prefill_kernel" in k]
    stores = [l.split()[0] for l in lines if l.strip().startswith(("global_store", "flat_store", "buffer_store", "scratch_store"))]
    assert stores == ["global_store_dwordx4"] * 16, stores
    # compiler-visible loads: the sixteen query loads at each of their two places, the sink (two forms, two places)
    loads = [l.split()[0] for l in lines if l.strip().startswith(("global_load", "flat_load", "buffer_load", "scratch_load"))
             and "_lds_" not in l]
    assert loads.count("global_load_dwordx4") == 32 and len(loads) == 36, loads


@pytest.mark.parametrize("source", ["sparse_attn.hip", "prefill_attn.hip", "flash_prefill.hip"])
def test_no_copy_into_lds_directly_follows_the_write_of_its_address_register(source):
    bodies = build.kernel_bodies(build.device_assembly(os.path.join(build.CSRC, source)))
    assert any("_load_lds_" in l for lines in bodies.values() for l in lines)
    for name, lines in bodies.items():
        assert build.m0_hazards(lines) == [], name
    copy = "\tglobal_load_lds_dwordx4 v2, s[4:5]"
    assert len(build.m0_hazards(["\ts_mov_b32 m0, s8", "\t;;#ASMSTART", copy])) == 1
    assert len(build.m0_hazards(["\ts_add_i32 m0, s8, 0x400", copy])) == 1
    assert build.m0_hazards(["\ts_mov_b32 m0, s8", "\ts_nop 0", copy, copy]) == []


@pytest.mark.parametrize("source", ["sparse_attn.hip", "prefill_attn.hip", "flash_prefill.hip", "topk.hip", "indexer.hip", "indexer_tiled.hip"])
def test_inline_asm_reads_no_scalar_register_too_soon(source):
    bodies = build.kernel_bodies(build.device_assembly(os.path.join(build.CSRC, source)))
    assert any("#ASMSTART" in l for lines in bodies.values() for l in lines)
    for name, lines in bodies.items():
        assert build.scalar_register_hazards(lines) == [], name
        # (the comparisons of the sampled top-k take no scalar operand at all, whatever the compiler puts in front of them)
        assert not any("v_cmp_le_i32_e64" in l and " s" in l.split(",", 1)[1] for l in _asm_lines(lines)), name
    compare = "\tv_cmp_le_i32_e64 s[2:3], s8, v1"
    for between, hazard in (([], 1), (["\ts_nop 0"], 1), (["\ts_nop 1"], 0), (["\tv_mov_b32_e32 v2, v3", "\ts_nop 0"], 0)):
        lines = ["\tv_readfirstlane_b32 s8, v0", *between, "\t;;#ASMSTART", compare, "\t;;#ASMEND"]
        assert len(build.scalar_register_hazards(lines)) == hazard
    copy = ["\t;;#ASMSTART", "\ts_mov_b32 m0, s4", "\ts_nop 0", "\tglobal_load_lds_dwordx4 v2, s[8:9]", "\t;;#ASMEND"]
    assert len(build.scalar_register_hazards(["\tv_readlane_b32 s9, v0, 3", "\ts_nop 1", *copy])) == 1
    assert build.scalar_register_hazards(["\tv_readlane_b32 s9, v0, 3", "\ts_nop 2", *copy]) == []
    assert build.scalar_register_hazards(["\tv_readlane_b32 s9, v0, 3", copy[3]]) == []  # (the compiler's own)
    carry = ["\t;;#ASMSTART", "\tv_addc_co_u32_e64 v1, vcc, v1, v1, s[2:3]", "\tv_addc_co_u32_e64 v1, vcc, v1, v1, s[4:5]"]
    assert build.scalar_register_hazards(carry) == []


def _asm_lines(lines):
    inside, out = False, []
    for line in lines:
        if "#ASMSTART" in line or "#ASMEND" in line:
            inside = "#ASMSTART" in line
        elif inside:
            out.append(line)
    return out


def test_scalar_arguments_of_kernels_are_preloaded():
    """The score, selection and rope kernels take plain arguments, which arrive in scalar registers with the wave."""
    for source, kernels in (("indexer_fp8.hip", 2), ("topk.hip", 22), ("rope_seam.hip", 9)):
        text = build.device_assembly(os.path.join(build.CSRC, source))
        lengths = [int(l.split()[1]) for l in text.splitlines() if l.strip().startswith(".amdhsa_user_sgpr_kernarg_preload_length")]
        assert len(lengths) == kernels and all(n >= 7 for n in lengths), (source, lengths)


@pytest.mark.parametrize("source,kernels", [("indexer.hip", 14), ("indexer_tiled.hip", 5)])
def test_scalar_arguments_of_the_other_score_kernels_are_preloaded(source, kernels):
    text = build.device_assembly(os.path.join(build.CSRC, source))
    lengths = [int(l.split()[1]) for l in text.splitlines() if l.strip().startswith(".amdhsa_user_sgpr_kernarg_preload_length")]
    assert len(lengths) == kernels and all(n >= 6 for n in lengths), lengths
