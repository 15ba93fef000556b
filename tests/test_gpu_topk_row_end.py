"""The sampled top-k at the end of a row: its last scores, for every remainder of four, in each number of threads."""

import numpy as np
import pytest
import torch

from moespresso_amd.runtime.deepseek_v4 import indexer_score_kernel as isk
from oracle import ds4

pytestmark = pytest.mark.gpu


# a first row of a piece and the rows up to the next four; one piece and none missing; strides of odd length
@pytest.mark.parametrize("rows,n,k", [(2, 2049, 64), (2, 4094, 512), (390, 2049, 64), (390, 5122, 512), (3, 8193, 512),
                                      (3, 16386, 1024), (3, 24577, 2048), (3, 28674, 2048), (3, 32763, 2048)])
@pytest.mark.parametrize("more", [0, 1, 2, 3])
def test_last_rows_are_selected(rows, n, k, more):
    n += more
    rng = np.random.default_rng(n)
    s = rng.standard_normal((3, n)).astype(np.float32)
    s[0, -5:] = 9.0 + np.arange(5)                       # the highest ones,
    s[1, -3:] = -np.inf                                  # the lowest ones,
    s[2, -7:] = 50.0                                     # and equal ones, more than are wanted of them
    s[2, : k - 4] = 60.0
    data = torch.from_numpy(s).cuda().repeat((rows + 2) // 3, 1)[:rows]
    got = isk.topk_select(data, k).cpu().numpy()
    for b in range(min(rows, 3)):
        want = ds4.radix_select_topk(s[b], k)
        np.testing.assert_array_equal(got[b], want)
        np.testing.assert_array_equal(got[rows - 1 - (rows - 1 - b) % 3], want)
