"""The native call path: operands that the path hands to Python."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_operands_outside_the_plain_case_give_the_same_results():
    from moespresso_amd.runtime.deepseek_v4 import attention_seam_kernel as seam
    from moespresso_amd.runtime.deepseek_v4 import indexer_score_kernel as isk

    scores = torch.randn((5, 3001), device="cuda")
    padded = torch.empty((5, 3100), device="cuda")
    padded[:, :3001] = scores
    assert isk.topk_select(padded[:, :3001], np.int64(512)).equal(isk.topk_select(scores, 512))
    x = torch.randn((1, 7, 3, 128), device="cuda").half()
    inv = torch.rand((32,), device="cuda")
    want = seam.fused_partial_rope(x, inv, offset=5)
    assert seam.fused_partial_rope(x.transpose(1, 2).contiguous().transpose(1, 2), inv, offset=5).equal(want)
    with pytest.raises(ValueError, match="topk must be positive"):
        isk.topk_select(scores, 3002)
    with pytest.raises(ValueError, match="partial-rope contract"):
        seam.fused_partial_rope(x, inv, offset=-1)
