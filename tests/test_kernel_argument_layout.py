"""Arguments that the attention kernels need at their start come in scalar registers with the wave, and their first requests to
memory wait for no others (CPU: hipcc compiles the source to assembly for gfx950, nothing runs)."""
import os
import re
import shutil

import pytest

from moespresso_amd import build

pytestmark = pytest.mark.skipif(not (os.path.exists(build.HIPCC) or shutil.which(build.HIPCC)), reason="hipcc not installed")


def _first_lines(lines, until):
    code = [l.split(";")[0].strip() for l in lines]
    code = [l for l in code if l and (not l.startswith(".") or l.endswith(":"))]
    start = next(i for i, l in enumerate(code) if l.startswith("s_branch"))  # (in front: the form for firmware that preloads nothing)
    code = code[start + 1:]
    return code[:next(i for i, l in enumerate(code) if re.match(until, l))]


def _preload_lengths(text):
    """Words of arguments that come in registers, of every kernel whose descriptor names a number."""
    found = {}
    for name, descriptor in re.findall(r"^\s*\.amdhsa_kernel (\S+)\n(.*?)^\s*\.end_amdhsa_kernel", text, flags=re.S | re.M):
        m = re.search(r"kernarg_preload_length (\d+)", descriptor)
        found[name] = int(m[1]) if m else 0
    return found


def test_a_kernel_without_a_preload_length_is_not_given_the_next_ones():
    text = ".amdhsa_kernel a\n.end_amdhsa_kernel\n.amdhsa_kernel b\n.amdhsa_user_sgpr_kernarg_preload_length 14\n.end_amdhsa_kernel\n"
    assert _preload_lengths(text) == {"a": 0, "b": 14}


def test_a_wait_is_seen_where_it_is_on_the_way():
    start = ["s_waitcnt lgkmcnt(0)", "s_branch .LBB0_0", ".LBB0_0:"]
    load, wait, copy, past = "s_load_dword s6, s[0:1], 0xd0", "s_waitcnt lgkmcnt(0)", "global_load_lds_dwordx4 v1, s[2:3]", "s_cbranch_scc1 .LBB0_1"
    for lines, waits in (([load, copy], 0), ([load, wait, copy], 1), ([load, past, wait, ".LBB0_1:", copy], 1),
                         ([past, load, wait, ".LBB0_1:", copy], 0), ([past, load, ".LBB0_1:", wait, copy], 1)):
        assert len(_waits_on_the_way(start + lines, r"global_load_lds")) == waits, lines


def _waits_on_the_way(lines, until):
    """Waits for arguments in front of the first instruction that matches `until`, but for those of blocks that load what they wait
    for themselves and that a conditional branch passes by."""
    found, passed_by, loads = [], False, False
    for line in _first_lines(lines, until):
        if line.startswith("s_cbranch"):
            passed_by, loads = True, False
        elif line.endswith(":"):
            passed_by = loads = False
        elif line.startswith("s_load"):
            loads = True
        elif line.startswith("s_waitcnt") and not (passed_by and loads):
            found.append(line)
    return found


# (the flash kernel's forms without an 8-bit prefix, whose tiles' addresses are in the struct)
@pytest.mark.parametrize("source,kernel,count", [("prefill_attn.hip", r"indexed_prefill_kernel", 4),
                                                 ("flash_prefill.hip", r"flash_prefill_kernelILi\dELb0", 10)])
def test_the_first_copies_wait_for_no_argument(source, kernel, count):
    text = build.device_assembly(os.path.join(build.CSRC, source))
    bodies = {k: v for k, v in build.kernel_bodies(text).items() if re.search(kernel, k)}
    assert len(bodies) == count
    for name, lines in bodies.items():
        assert _waits_on_the_way(lines, r"global_load_lds") == [], name


def test_the_split_kernel_requests_its_ids_before_it_waits_for_an_argument():
    text = build.device_assembly(os.path.join(build.CSRC, "sparse_attn.hip"))
    bodies = {k: v for k, v in build.kernel_bodies(text).items() if "sparse_attn_split_kernel" in k}
    assert len(bodies) == 6
    for name, lines in bodies.items():
        head = _first_lines(lines, r"global_load_dword v")
        assert not any(l.startswith("s_waitcnt") for l in head), name
    lengths = _preload_lengths(text)
    assert sum("split_kernel" in k for k in lengths) == 6 and sum("merge_kernel" in k for k in lengths) == 3
    assert all(n >= 11 for k, n in lengths.items() if "split_kernel" in k or "merge_kernel" in k), lengths


def test_the_8_bit_split_requests_its_first_tiles_before_it_waits_for_an_argument():
    """A tile is eight 16-byte loads a lane of K codes and eight of V codes. (The first of them, and what they wait for, is one
    basic block: a wave without a tile branches around it.)"""
    text = build.device_assembly(os.path.join(build.CSRC, "q8_decode.hip"))
    bodies = {k: v for k, v in build.kernel_bodies(text).items() if "q8_decode_split_kernel" in k}
    assert len(bodies) == 6
    for name, lines in bodies.items():
        head = _first_lines(lines, r"s_waitcnt")
        assert sum(l.startswith("global_load_dwordx4 ") for l in head) >= 16, name


def _argument_bytes(text):
    """Size of every kernel's argument block, hidden arguments included."""
    records = re.split(r"\n  - \.", text[text.index("amdhsa.kernels:"):])[1:]
    return {re.search(r"\.name:\s+(_Z\S+)", r)[1]: int(re.search(r"\.kernarg_segment_size:\s+(\d+)", r)[1]) for r in records}


# (a call that the host issues more slowly than the device runs it pays for long blocks)
@pytest.mark.parametrize("source,kernel,count,most", [("sparse_attn.hip", "sparse_attn_split_kernel", 6, 312),
                                                      ("sparse_attn.hip", "sparse_attn_merge_kernel", 3, 112),
                                                      ("prefill_attn.hip", "indexed_prefill_kernel", 4, 136),
                                                      ("flash_prefill.hip", "flash_prefill_kernelILi.ELb0", 10, 88),
                                                      ("flash_prefill.hip", "flash_prefill_kernelILi.ELb1", 18, 152),
                                                      ("q8_decode.hip", "q8_decode_split_kernel", 6, 104)])
def test_argument_blocks_hold_no_field_twice(source, kernel, count, most):
    sizes = [n for name, n in _argument_bytes(build.device_assembly(os.path.join(build.CSRC, source))).items() if re.search(kernel, name)]
    assert len(sizes) == count and max(sizes) <= most, sizes
