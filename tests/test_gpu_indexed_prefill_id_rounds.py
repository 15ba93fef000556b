"""The prefill attention kernel's id staging: two rounds of 256 ids are requested ahead of the queries where a single
round of units is cut into ranges, none elsewhere."""

import numpy as np
import pytest
import torch

from oracle import ds4

pytestmark = pytest.mark.gpu


# the last id of a round, the first of the next, the first that is not requested ahead, and the lengths around both lines; in
# each, the walk ends at a different place for every token or (first token's position 0) at the first id
@pytest.mark.parametrize("tokens,top_k", [(5, 1), (5, 255), (5, 256), (5, 257), (5, 512), (5, 513), (5, 800), (512, 257), (513, 257)])
@pytest.mark.parametrize("pos0", [0, 2900])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_rounds_match_the_oracle(tokens, top_k, pos0, dtype):
    from moespresso_amd.runtime.deepseek_v4 import indexed_attention_kernel as iak

    gen = torch.Generator(device="cuda").manual_seed(top_k)
    heads, pool = 8, 900
    q = torch.randn((1, heads, tokens, 512), device="cuda", generator=gen).to(dtype)
    raw = torch.randn((1, 1, min(127, pos0) + tokens, 512), device="cuda", generator=gen).half()
    comp = torch.randn((1, pool, 512), device="cuda", generator=gen).half()
    ids = torch.rand((1, tokens, pool), device="cuda", generator=gen).topk(top_k, dim=2).indices.to(torch.int32)
    ids = torch.where(ids >= 725, torch.minimum(ids, torch.full_like(ids, 724)), ids)  # the first token of 2900 sees 725 rows
    t = torch.arange(tokens, device="cuda")
    ids[0, t, (t * 263) % top_k] = pool - 1  # and ends its walk here
    sinks = torch.randn(heads, device="cuda", generator=gen)
    run = iak.indexed_mixed_attention_prefill_live_f16 if dtype == torch.float16 else iak.indexed_mixed_attention_prefill_live_f32
    got = run(q, raw, comp, ids, sinks, pos0=pos0, window=128, ratio=4)
    want = ds4.indexed_mixed_attention_prefill(q[0].transpose(0, 1).float().cpu().numpy(), raw[0, 0].cpu().numpy(), comp[0].cpu().numpy(),
                                               ids[0].cpu().numpy(), sinks.cpu().numpy(), pos0=pos0, window=128, ratio=4)
    np.testing.assert_allclose(got[0].transpose(0, 1).cpu().numpy(), want, rtol=2e-3, atol=2e-3)
