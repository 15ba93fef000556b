"""The native call path: quantise-on-append into a cache's own buffers, and operands that the path hands to Python."""

import numpy as np
import pytest
import torch

from oracle import qwen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("batch,heads,width,chunks", [(1, 2, 256, (255, 1, 1)), (3, 1, 64, (1, 260)), (2, 4, 320, (37, 219, 5))])
def test_append_writes_the_rows_of_every_head_behind_the_prefix(dtype, batch, heads, width, chunks):
    from moespresso_amd.runtime.qwen import kquant

    gen = torch.Generator(device="cuda").manual_seed(7)
    cache, rows = kquant.QuantizedKVCache(), []
    for n in chunks:
        kv = [torch.randn((batch, heads, n, width), device="cuda", generator=gen).to(dtype) for _ in range(2)]
        rows.append(kv)
        k, v = cache.update_and_fetch(*kv)
    for side, i in ((k, 0), (v, 1)):
        x = torch.cat([r[i] for r in rows], dim=2)
        want = qwen.affine_q8_quantize(x.float().cpu().numpy())
        assert side[0].shape[2] == sum(chunks)
        np.testing.assert_array_equal(side[0].contiguous().view(torch.int32).cpu().numpy().view(np.uint32), want[0])
        for got, ref in zip(side[1:], want[1:]):
            torch.testing.assert_close(got.cpu(), torch.from_numpy(ref).to(dtype), rtol=0, atol=0)


def test_append_of_a_transposed_view_and_of_another_type_goes_through_the_copy():
    from moespresso_amd.runtime.qwen import kquant

    x = torch.randn((1, 9, 2, 256), device="cuda")
    views, dense = kquant.QuantizedKVCache(), kquant.QuantizedKVCache()
    views.update_and_fetch(x.transpose(1, 2), x.transpose(1, 2))
    dense.update_and_fetch(x.transpose(1, 2).contiguous(), x.transpose(1, 2).contiguous())
    views.update_and_fetch(x[:, :1].half().transpose(1, 2), x[:, :1].half().transpose(1, 2))
    dense.update_and_fetch(x[:, :1].half().float().transpose(1, 2), x[:, :1].half().float().transpose(1, 2))
    for a, b in zip(views.state[0] + views.state[1], dense.state[0] + dense.state[1]):
        assert a.shape == b.shape
        codes = a.dtype == torch.uint32
        assert codes or a[:, :, :9].equal(b[:, :, :9])
        assert not codes or a.view(torch.int32)[:, :, :].equal(b.view(torch.int32))


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
