"""Arguments that sparse attention's split and merge kernels need at their start come in scalar registers with the wave (CPU:
hipcc compiles the source to assembly for gfx950, nothing runs)."""
import os
import re
import shutil

import pytest

from moespresso_amd import build

pytestmark = pytest.mark.skipif(not (os.path.exists(build.HIPCC) or shutil.which(build.HIPCC)), reason="hipcc not installed")


def _first_lines(lines, until):
    code = [l.split(";")[0].strip() for l in lines]
    code = [l for l in code if l and not l.startswith(".")]
    start = next(i for i, l in enumerate(code) if l.startswith("s_branch"))  # (in front: the form for firmware that preloads nothing)
    end = next(i for i, l in enumerate(code) if re.match(until, l))
    return code[start + 1:end]


def test_the_split_kernel_requests_its_ids_before_it_waits_for_an_argument():
    text = build.device_assembly(os.path.join(build.CSRC, "sparse_attn.hip"))
    bodies = {k: v for k, v in build.kernel_bodies(text).items() if "sparse_attn_split_kernel" in k}
    assert len(bodies) == 6
    for name, lines in bodies.items():
        head = _first_lines(lines, r"global_load_dword v")
        assert not any(l.startswith("s_waitcnt") for l in head), name
    preload = dict(re.findall(r"\.amdhsa_kernel (\S+).*?kernarg_preload_length (\d+)", text, flags=re.S))
    assert all(int(n) >= 11 for k, n in preload.items() if "split_kernel" in k or "merge_kernel" in k)
