"""Top-k of rows whose wanted part is small (selected from the keys above a sampled pivot): widths around the kernel's pieces,
few and many rows, a start off 16 bytes, and rows whose sample says little about the row."""
import numpy as np
import pytest
import torch

from moespresso_amd.runtime.deepseek_v4 import indexer_score_kernel as isk
from oracle import ds4

pytestmark = pytest.mark.gpu


def rows_of(kinds, n, k, rng):
    s = rng.standard_normal((kinds, n)).astype(np.float32)
    s[0] = np.abs(s[0]) * 3 + 20                         # as scores are: positive, one binade
    s[1] -= 50                                           # a pivot below zero
    s[2, n // 3:] = -np.inf                              # rows a token does not see
    s[2, 5], s[2, 7], s[2, 9] = np.inf, np.nan, -np.float32(np.nan)
    s[3] = np.round(s[3] * 4)                            # ties, -0 among them, at the k-th key
    s[4] = np.float32(0.25)                              # one value
    s[5] = np.linspace(0, 1, n, dtype=np.float32) + s[5] * 1e-3
    s[6] = s[6] * 1e-3 + 1
    s[6, 3] = 1e30                                       # one bin holds the row
    s[7] = np.where(np.arange(n) % 4 == 1, s[7] + 100, s[7])   # the wanted rows at one place of every piece
    s[8, n - k:] += 1000                                 # all of them at the row's end
    return s


@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("n,k", [(2049, 1), (2051, 768), (3072, 512), (3073, 64), (4096, 1536), (4097, 512), (6145, 3000),
                                 (8192, 2048), (8193, 512), (12289, 1024), (20481, 4000), (28673, 2048), (32767, 1),
                                 (32768, 2048)])
def test_topk_from_a_sampled_pivot(n, k, many):
    rng = np.random.default_rng(n + k)
    s = rows_of(9, n, k, rng)
    data = torch.from_numpy(s).cuda()
    if many:
        data = data.repeat(43, 1)                        # 387 rows
    wide = torch.zeros((data.shape[0], n + 3), device="cuda")   # rows one element off
    wide[:, 1:n + 1] = data
    got = isk.topk_select(data, k).cpu().numpy()
    off = isk.topk_select(wide[:, 1:n + 1], k).cpu().numpy()
    for b in range(9):
        want = ds4.radix_select_topk(s[b], k)
        np.testing.assert_array_equal(got[b], want)
        np.testing.assert_array_equal(off[b], want)
        np.testing.assert_array_equal(got[-9 + b], want)
