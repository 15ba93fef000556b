"""Query QAT where the group scale is, and is not, exactly a power of two, and score rows at the edges of how pool tiles
are dealt to workgroups."""
import numpy as np
import pytest
import torch

from oracle import ds4
from moespresso_amd.runtime.deepseek_v4 import indexer_score_kernel as isk

pytestmark = pytest.mark.gpu


# exponents of the group scales; the table's entry is the power of two itself from -12 to 12 only
@pytest.mark.parametrize("low,high", [(-12, 12), (-14, -12), (13, 16), (-66, -60), (58, 68)])
def test_qat_rows_of_mixed_scales_bitexact(low, high):
    rng = np.random.default_rng(high + 100)
    rows = rng.standard_normal((257, 128)).astype(np.float32)
    # one Hadamard basis row a line: every rotated value is +-1 times the row's factor, so lattice midpoints occur
    signs = np.array([[1.0 - 2.0 * (bin(i & j).count("1") & 1) for j in range(128)] for i in (0, 3, 77, 127)], np.float32)
    mids = np.array([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0, 6.0], np.float32)
    rows[:32] = (mids[:, None, None] * signs[None]).reshape(32, 128)
    rows *= np.exp2(rng.integers(low, high + 1, (257, 1))).astype(np.float32)
    rows[40, :64] = -0.0
    got = isk.indexer_qat_rows(torch.from_numpy(rows).cuda()).cpu().numpy()
    np.testing.assert_array_equal(got.view(np.uint32), ds4.indexer_qat(rows).view(np.uint32))


# a workgroup for each tile, the last of them; one more tile than 256 workgroups; the first row count of 257 workgroups
@pytest.mark.parametrize("n_rows", [1, 33, 256 * 32, 256 * 32 + 1, 2048 * 32, 2048 * 32 + 1])
def test_score_row_at_the_edges_of_the_split(n_rows):
    rng = np.random.default_rng(n_rows)
    q = rng.standard_normal((1, 64, 1, 128), dtype=np.float32)
    pooled = ds4.indexer_qat(rng.standard_normal((1, n_rows, 128), dtype=np.float32))
    w = (rng.standard_normal((1, 1, 64), dtype=np.float32) / 8).astype(np.float32)
    got = isk.fused_qat_indexer_scores(*(torch.from_numpy(a).cuda() for a in (q, pooled, w)), 128 ** -0.5).cpu().numpy()
    np.testing.assert_allclose(got, ds4.fused_qat_indexer_scores(q, pooled, w, 128 ** -0.5), rtol=1e-5, atol=1e-5)
