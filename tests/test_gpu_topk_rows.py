"""Top-k of rows of up to 8192 scores at the widths of the kernel, with values that move its bins: rows mostly -inf (with
more wanted than finite scores), NaN of both signs, one huge value over close ones, a k-th key inside ties."""
import numpy as np
import pytest
import torch

from moespresso_amd.runtime.deepseek_v4 import indexer_score_kernel as isk
from oracle import ds4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [5, 257])  # 257: past one row per compute unit
@pytest.mark.parametrize("n,k", [(1, 1), (513, 512), (1024, 513), (1025, 64), (2048, 1), (2049, 2049), (3072, 512),
                                 (3073, 1025), (4096, 2048), (4095, 4000), (4097, 512), (8192, 2049)])
def test_topk_rows(rows, n, k):
    rng = np.random.default_rng(n + k + rows)
    s = rng.standard_normal((rows, n)).astype(np.float32)
    s[1, min(n, k) // 2:] = -np.inf                      # fewer finite scores than wanted
    s[2] = np.float32(1.0) + rng.random(n).astype(np.float32) * np.float32(1e-5)
    s[2, 0] = 3e38                                       # one bin holds nearly all of the row
    s[3] = np.round(s[3] * 2) / 2                        # ties
    s[4, ::3] = -np.inf
    s[4, 1::5] = -np.float32(np.nan)                     # below -inf
    s[4, 2::7] = np.nan                                  # above inf
    got = isk.topk_select(torch.from_numpy(s).cuda(), k).cpu().numpy()
    for b in (0, 1, 2, 3, 4, rows - 1):
        np.testing.assert_array_equal(got[b], ds4.radix_select_topk(s[b], k))
