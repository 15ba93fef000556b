"""The wide form of the partial rope where it can go wrong: part-filled blocks of positions, outer rows that do not fill a
slab, widths at both ends of its range and just outside."""

import numpy as np
import pytest
import torch

from moespresso_amd.runtime.deepseek_v4 import attention_seam_kernel as seam
from oracle import ds4

pytestmark = pytest.mark.gpu
_TORCH = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}


@pytest.mark.parametrize("dtype_name", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("shape", [(1, 32, 64), (5, 33, 64), (3, 17, 128), (4, 9, 256), (7, 5, 512), (9, 4, 512), (5, 3, 1024),
                                   (2, 4, 2048), (6, 40, 96)])
def test_rows_bit_identical(dtype_name, shape):
    rng = np.random.default_rng(shape[0] + shape[2])
    x = torch.from_numpy((2.0 * rng.standard_normal(shape)).astype(np.float32)).to(_TORCH[dtype_name])
    inv = ds4.rope_inverse_frequencies(64, 10000.0).astype(np.float32)
    for inverse, offset, positions in ((False, 3855, None), (True, 0, rng.permutation(9000)[:shape[1]].astype(np.float32))):
        got = seam.fused_partial_rope(x.cuda(), torch.from_numpy(inv).cuda(), offset=offset, inverse=inverse,
                                      positions=None if positions is None else torch.from_numpy(positions).cuda())
        want = ds4.fused_partial_rope(x.float().numpy(), inv, offset=offset, inverse=inverse, positions=positions, dtype=dtype_name)
        bits = torch.int32 if dtype_name == "float32" else torch.int16
        assert got.cpu().view(bits).equal(torch.from_numpy(want).to(_TORCH[dtype_name]).view(bits))


@pytest.mark.parametrize("dtype_name", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("inverse", [False, True])
def test_rows_past_the_caches_are_those_of_smaller_calls(dtype_name, inverse):
    gen = torch.Generator(device="cuda").manual_seed(4)
    x = torch.randn((65, 3027, 128), device="cuda", generator=gen).to(_TORCH[dtype_name])    # 24.02 M elements
    inv = torch.from_numpy(ds4.rope_inverse_frequencies(64, 10000.0).astype(np.float32)).cuda()
    got = seam.fused_partial_rope(x, inv, offset=71, inverse=inverse)
    for part, want in ((x[:32], got[:32]), (x[32:], got[32:])):
        assert seam.fused_partial_rope(part, inv, offset=71, inverse=inverse).equal(want)
