"""Tiled scores over few tokens: each way of dealing the pool rows out to workgroups (4, 8 or 16 pairs of tiles at least), with
operands of the fp4 format, operands that are not, and one token block among others that is not."""
import pytest
import torch

from test_gpu_tiled_scores_fp4 import _both, _operands

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spoil", ["no", "all", "one token"])
@pytest.mark.parametrize("batch,tokens,rows", [(1, 96, 2000), (1, 67, 4001), (2, 300, 610), (1, 1000, 500), (1, 517, 2053),
                                               (1, 2, 65537), (1, 129, 1023)])
def test_rows_are_dealt_out_whatever_the_operands_are(batch, tokens, rows, spoil):
    q, w, comp = _operands(batch, 64, tokens, rows, torch.float32)
    if spoil == "all":
        q, comp = q + 0.03125, comp - 0.015625
    elif spoil == "one token":
        q[-1, 17, tokens // 2, 5] += 0.03125
    got, want = _both(q, w, comp, 4 * rows - tokens // 2)
    assert got.equal(want)
