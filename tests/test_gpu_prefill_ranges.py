"""Chunked prefill over few and many key ranges (each merge form), and both ways to read a quantised prefix."""
import numpy as np
import pytest
import torch

from moespresso_amd.runtime.qwen import kquant
from oracle import qwen

pytestmark = pytest.mark.gpu


# ranges of two tiles; of more than 32 (four waves a merged row); 9 to 16; at most 8; the last workgroup of rows ragged
@pytest.mark.parametrize("heads,kv_heads,tokens,past", [(16, 2, 33, 100), (4, 1, 17, 5000), (16, 2, 33, 9001),
                                                       (16, 2, 203, 2000), (2, 1, 389, 3000), (16, 2, 700, 500)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_flash_prefill_ranges(heads, kv_heads, tokens, past, dtype):
    gen = torch.Generator().manual_seed(tokens)
    q, k, v = (torch.randn(s, generator=gen).mul(0.5).to(dtype) for s in
               ((1, heads, tokens, 256), (1, kv_heads, past + tokens, 256), (1, kv_heads, past + tokens, 256)))
    got = kquant.flash_prefill(q.cuda(), k.cuda(), v.cuda(), 256 ** -0.5, past_len=past).float().cpu().numpy()
    want = qwen.causal_prefill_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(), 256 ** -0.5, past=past)
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert (np.abs(got - want) <= 2e-3 + ulp * np.abs(want)).all()


# 128 tokens: unpacked in the attention kernel, 129: rows converted first; prefixes of whole and ragged tiles and rows
@pytest.mark.parametrize("tokens", [128, 129, 1023])
@pytest.mark.parametrize("past", [0, 31, 32, 305])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_quantised_prefix_rows(tokens, past, dtype):
    gen = torch.Generator(device="cuda").manual_seed(tokens + past)
    q, k, v = (torch.randn((1, h, past + tokens, 256), device="cuda", generator=gen).mul_(0.1).to(dtype) for h in (8, 2, 2))
    tk, tv = kquant.quantize(k), kquant.quantize(v)
    dk, dv = kquant.dequantize(*tk), kquant.dequantize(*tv)
    prefix = [t[:, :, :past] for t in (*tk, *tv)]
    got = kquant.sdpa_fa_prefill_q8(q[:, :, past:].float(), *prefix, dk[:, :, past:], dv[:, :, past:], 256 ** -0.5)
    want = qwen.causal_prefill_attention(q[:, :, past:].float().cpu().numpy(), dk.float().cpu().numpy(),
                                         dv.float().cpu().numpy(), 256 ** -0.5, past=past)
    assert np.abs(got.cpu().numpy() - want).max() < 2e-3
