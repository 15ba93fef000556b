"""Decode attention where the waves of a workgroup differ: head counts that leave waves without heads or with some, and single
keys that outgrow the running maximum of one head, in every eighth-of-keys share of a tile and in early and late tiles."""
import numpy as np
import pytest
import torch

from moespresso_amd.runtime.deepseek_v4 import indexed_attention_kernel as iak
from oracle import ds4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,spike", [(torch.float16, 14.0), (torch.bfloat16, 80.0)])
@pytest.mark.parametrize("heads,k_dim,batch,ids", [(1, 512, 3, 200), (31, 576, 2, 70), (33, 512, 1, 500), (64, 576, 40, 250),
                                                   (65, 576, 2, 96), (100, 512, 300, 64)])
def test_single_keys_outgrow_the_maximum(dtype, spike, heads, k_dim, batch, ids):
    gen = torch.Generator(device="cuda").manual_seed(heads + ids)
    rng = np.random.default_rng(heads)
    scale = k_dim ** -0.5
    q = torch.randn((batch, heads, k_dim), device="cuda", generator=gen).to(dtype)
    kv = torch.randn((batch, ids + 20, k_dim), device="cuda", generator=gen)
    # every 8 + 32 n +- a few keys, one row points along one head's query: logit of `spike` log2 units or more above the rest
    qf = q.float()
    for j, row in enumerate(range(3, ids, 27)):
        h = int(rng.integers(0, heads))
        direction = qf[:, h] / qf[:, h].norm(dim=1, keepdim=True)
        kv[:, row] = direction * ((spike * (1 + 0.3 * j)) / (1.4427 * scale) / qf[:, h].norm(dim=1, keepdim=True))
    kv = kv.to(dtype)
    sel = torch.arange(ids, dtype=torch.int32, device="cuda").expand(batch, ids).contiguous()
    sinks = torch.randn((heads,), device="cuda", generator=gen)
    got = iak.sparse_mla_decode(q, kv, sel, scale=scale, window_start=ids, window_rows=20, sinks=sinks).float().cpu().numpy()
    pick = [0, batch - 1]
    rows = np.tile(np.concatenate([np.arange(ids, ids + 20), np.arange(ids)]), (2, 1))
    qr, kvr = q.float().cpu().numpy()[pick], kv.float().cpu().numpy()[pick]
    want = ds4.sparse_mla_decode(qr, kvr, rows, scale=scale, sinks=sinks.cpu().numpy())
    # 2e-3, and three roundings (weights, partials, output) of the attention over |V|
    eps = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    logits = np.einsum("bhd,bnd->bhn", qr.astype(np.float64), kvr[:, rows[0]].astype(np.float64)) * scale
    logits = np.concatenate([logits, np.broadcast_to(sinks.cpu().numpy()[None, :, None], logits.shape[:2] + (1,))], axis=2)
    p = np.exp(logits - logits.max(axis=2, keepdims=True))
    p /= p.sum(axis=2, keepdims=True)
    mass = p[..., :-1] @ np.abs(kvr[:, rows[0], :512].astype(np.float64))
    assert np.isfinite(got).all()
    assert (np.abs(got[pick] - want) <= 2e-3 + 3 * eps * mass).all(), (np.abs(got[pick] - want) - 3 * eps * mass).max()


@pytest.mark.parametrize("window,ids", [(16, 16), (32, 32), (32, 64), (64, 65), (128, 300)])  # one tile each, 2, 3, 5 and 14 ranges
def test_rotated_decode_with_few_key_ranges(window, ids):
    from moespresso_amd.runtime.deepseek_v4 import decode_attention_kernel as dak

    rng = np.random.default_rng(window + ids)
    q, ring = (rng.standard_normal(s).astype(np.float16) for s in ((64, 512), (window, 512)))
    row, pooled = (rng.standard_normal(s).astype(np.float16) for s in (512, (400, 512)))
    sel = np.sort(rng.choice(400, ids, replace=False)).astype(np.int32)
    sinks = rng.standard_normal(64).astype(np.float16)
    inv = ds4.rope_inverse_frequencies(64, ds4.DS4_COMPRESS_ROPE_BASE, ds4.DS4_YARN).astype(np.float32)
    params = np.array([12345, 5], dtype=np.int32)
    got = dak.fused_decode_sdpa(*(torch.from_numpy(x).cuda() for x in (q, ring, row, pooled, sel, sinks, inv, params)),
                                scale=512 ** -0.5).float().cpu().numpy()
    want = ds4.fused_decode_sdpa(q, ring, row, pooled, sel, sinks, inv, params, scale=512 ** -0.5).astype(np.float32)
    # weights, partial, output and the three roundings of the rotation in float16, of values of at most max |V|
    bound = 2e-3 + 6 * 2.0 ** -11 * max(np.abs(ring).max(), np.abs(row).max(), np.abs(pooled).max())
    assert np.abs(got - want).max() <= bound
