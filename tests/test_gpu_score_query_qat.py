"""The query QAT inside the score row: one head's weight and one-hot pool rows show every prepared query value, at lattice
midpoints, next to them, and at group scales inside and outside the range that is converted directly."""
import numpy as np
import pytest
import torch

from moespresso_amd.runtime.deepseek_v4 import indexer_score_kernel as isk
from oracle import ds4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("low,high", [(0, 0), (-10, 10), (-16, 16), (-40, -14)])
@pytest.mark.parametrize("heads", [64, 37])
def test_prepared_queries_are_those_of_the_row_operator(heads, low, high):
    rng = np.random.default_rng(high + heads)
    q = rng.standard_normal((heads, 128)).astype(np.float32)
    # one Hadamard basis row a line: every rotated value is +-1 times the row's factor
    signs = np.array([[1.0 - 2.0 * (bin(i & j).count("1") & 1) for j in range(128)] for i in (0, 3, 77, 127)], np.float32)
    mids = np.array([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0, 6.0], np.float32)
    q[:32] = (mids[:, None, None] * signs[None]).reshape(32, 128)
    q[32] = 0.0
    q[33, :64] = -0.0
    # groups of midpoints: what the rotation of these rows gives, up to the rounding of its sums
    for i, ulps in ((34, 0), (35, 1), (36, -1)):
        target = np.tile(np.concatenate([mids, -mids]), 8).astype(np.float32)
        target = (target.view(np.int32) + ulps).view(np.float32)
        h = np.array([[1.0 - 2.0 * (bin(a & b).count("1") & 1) for b in range(128)] for a in range(128)])
        q[i] = (h @ target.astype(np.float64) * 128 ** -0.5).astype(np.float32)
    q *= np.exp2(rng.integers(low, high + 1, (heads, 1))).astype(np.float32)
    pooled = np.concatenate([np.eye(128, dtype=np.float32), -np.eye(128, dtype=np.float32)])
    want = ds4.indexer_qat(q)
    picked = range(0, heads, 5)
    for h in (*range(36), *picked) if heads == 37 else (32, 33, 34, 35, 36, *picked):
        w = np.zeros((1, 1, heads), np.float32)
        w[0, 0, h] = 1.0
        got = isk.fused_qat_indexer_scores(torch.from_numpy(q[None, :, None]).cuda(), torch.from_numpy(pooled[None]).cuda(),
                                           torch.from_numpy(w).cuda(), 1.0).cpu().numpy().reshape(256)
        np.testing.assert_array_equal(got[:128] - got[128:], want[h], err_msg=str(h))


@pytest.mark.parametrize("outsider", [0, 9, 36, 63])
def test_one_head_outside_the_direct_range(outsider):
    """One wave's rows cannot be converted directly: all of the workgroup's are taken in float32 form, the ones already
    written as bfloat16 numbers among them."""
    rng = np.random.default_rng(outsider)
    q = rng.standard_normal((64, 128)).astype(np.float32)
    q[outsider] *= np.float32(2.0 ** 20)
    pooled = np.concatenate([np.eye(128, dtype=np.float32), -np.eye(128, dtype=np.float32)])
    want = ds4.indexer_qat(q)
    for h in (0, 1, 7, 8, 9, 35, 36, 56, 63):
        w = np.zeros((1, 1, 64), np.float32)
        w[0, 0, h] = 1.0
        got = isk.fused_qat_indexer_scores(torch.from_numpy(q[None, :, None]).cuda(), torch.from_numpy(pooled[None]).cuda(),
                                           torch.from_numpy(w).cuda(), 1.0).cpu().numpy().reshape(256)
        np.testing.assert_array_equal(got[:128] - got[128:], want[h], err_msg=str(h))
