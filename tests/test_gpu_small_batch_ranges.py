"""Decode attention of few sequences, where a key range is whole tiles of the window and then of the ids."""
import numpy as np
import pytest
import torch

from oracle import ds4
from moespresso_amd.runtime.deepseek_v4 import indexed_attention_kernel as iak

pytestmark = pytest.mark.gpu


# (batch, window, ids): one id; a tile each; window tile alone in a range; ragged window and ids; the last range ragged;
# a range that starts in the window and ends in the ids; two tiles a range; no window
@pytest.mark.parametrize("batch,window,ids", [(1, 1, 1), (1, 32, 32), (1, 33, 640), (2, 97, 513), (1, 128, 2047),
                                              (5, 100, 1985), (1, 128, 2048), (3, 0, 1200), (8, 31, 2000)])
def test_decode_ranges_of_whole_tiles(batch, window, ids):
    rng = np.random.default_rng(window + ids)
    n = 9000
    gen = torch.Generator(device="cuda").manual_seed(ids)
    kv = torch.randn((batch, n, 512), device="cuda", generator=gen).to(torch.bfloat16)
    q = torch.randn((batch, 64, 512), device="cuda", generator=gen).to(torch.bfloat16)
    sel = np.stack([rng.choice((n - window) // 4, ids, replace=False) for _ in range(batch)]).astype(np.int32)
    got = iak.sparse_mla_decode(q, kv, torch.from_numpy(sel).cuda(), scale=512 ** -0.5, window_start=n - window,
                                window_rows=window, row_mul=4, row_add=3).float().cpu().numpy()
    rows = np.concatenate([np.tile(np.arange(n - window, n), (batch, 1)), 4 * sel + 3], axis=1)
    gathered = np.stack([kv[b].float().cpu().numpy()[rows[b]] for b in range(batch)])
    local = np.tile(np.arange(rows.shape[1]), (batch, 1))
    want = ds4.sparse_mla_decode(q.float().cpu().numpy(), gathered, local, scale=512 ** -0.5, sinks=None)
    # the operator's bar: 2e-3, and the unit roundoff of a bfloat16 output (2^-8)
    bound = 2e-3 + 2.0 ** -8 * np.abs(want)
    if window + ids < 32:
        # the weights are bfloat16 too, which does not average out over so few keys: 2^-8 of the attention over |V|
        logits = q.double().cpu().numpy() @ gathered.astype(np.float64).transpose(0, 2, 1) * 512 ** -0.5
        weights = np.exp(logits - logits.max(axis=2, keepdims=True))
        bound = 2.0 ** -8 * (weights / weights.sum(axis=2, keepdims=True) @ np.abs(gathered)) + 2.0 ** -8 * np.abs(want)
    assert (np.abs(got - want) <= bound).all(), (np.abs(got - want) - bound).max()


@pytest.mark.parametrize("ids", [20, 2000])          # one key range, written directly; many, merged
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_a_row_that_is_not_finite_makes_its_columns_nan(ids, dtype):
    """An infinite element whose score is -inf has weight zero, and zero times infinity is NaN in that column alone; a score
    of +inf makes the whole row NaN. A partial stored as float16 must not turn either into a finite value."""
    gen = torch.Generator(device="cuda").manual_seed(ids)
    kv = torch.randn((2, 4000, 512), device="cuda", generator=gen).to(dtype)
    q = torch.randn((2, 64, 512), device="cuda", generator=gen).to(dtype)
    sel = torch.arange(ids, dtype=torch.int32, device="cuda").expand(2, ids).contiguous()
    kv[1, ids // 2, 300] = float("inf")
    q[1, :, 300] = torch.where(torch.arange(64, device="cuda") % 2 == 0, -1.0, 1.0).to(dtype)
    got = iak.sparse_mla_decode(q, kv, sel, scale=512 ** -0.5)
    want = torch.zeros((2, 64, 512), dtype=torch.bool, device="cuda")
    want[1, 0::2, 300] = True
    want[1, 1::2] = True
    assert got.isnan().equal(want) and bool(got[~want].isfinite().all())
