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


# Both sides of the line between unpacking in the attention kernel and converting beforehand, for four, five, one and six
# workgroups to a tile; 1023 and 1024 tokens of one query head to a KV head (unpacked, and converted to bfloat16)
@pytest.mark.parametrize("heads,kv_heads,tokens,past", [
    (4, 1, 200, 16384), (4, 1, 200, 16385), (4, 1, 256, 16400), (4, 1, 257, 16400), (2, 2, 130, 2048), (2, 2, 130, 2049),
    (16, 2, 150, 12288), (16, 2, 150, 12289), (3, 3, 1023, 6000), (3, 3, 1024, 6000)])
def test_quantised_prefix_at_the_line_between_unpacking_and_conversion(heads, kv_heads, tokens, past):
    gen = torch.Generator(device="cuda").manual_seed(past)
    q, k, v = (torch.randn((1, h, past + tokens, 256), device="cuda", generator=gen).mul_(0.1) for h in (heads, kv_heads, kv_heads))
    tk, tv = kquant.quantize(k), kquant.quantize(v)
    dk, dv = kquant.dequantize(*tk), kquant.dequantize(*tv)
    prefix = [t[:, :, :past] for t in (*tk, *tv)]
    got = kquant.sdpa_fa_prefill_q8(q[:, :, past:], *prefix, dk[:, :, past:], dv[:, :, past:], 256 ** -0.5)
    want = qwen.causal_prefill_attention(q[:, :, past:].cpu().numpy(), dk.cpu().numpy(), dv.cpu().numpy(), 256 ** -0.5, past=past)
    assert np.abs(got.cpu().numpy() - want).max() < 2e-3


# unpacked in the attention kernel; converted to float16; to bfloat16: one key range, several, and merges of two waves a row
@pytest.mark.parametrize("tokens,past", [(17, 40), (17, 5000), (203, 301), (300, 9000), (1024, 70)])
@pytest.mark.parametrize("side", ["key", "value"])
@pytest.mark.parametrize("bad", ["infinite activation", "infinite bias", "NaN scale"])
def test_infinities_and_nan_of_a_quantised_prefix_reach_the_output(tokens, past, side, bad):
    """As in decode over the same cache: a key that is not a number makes its KV head's rows NaN, a value its group's columns."""
    gen = torch.Generator(device="cuda").manual_seed(tokens + past)
    q, k, v = (torch.randn((1, h, past + tokens, 256), device="cuda", generator=gen).mul_(0.1) for h in (8, 2, 2))
    dirty_k, dirty_v = k.clone(), v.clone()
    at = (0, 1, past // 2)                                               # second head
    if bad == "infinite activation":
        (dirty_k if side == "key" else dirty_v)[(*at, 70)] = float("inf")  # second group: columns 64 to 127
    prefix = [t[:, :, :past] for t in (*kquant.quantize(dirty_k), *kquant.quantize(dirty_v))]
    scales, biases = prefix[1:3] if side == "key" else prefix[4:6]
    if bad == "infinite bias":
        biases[(*at, 1)] = float("inf")
    elif bad == "NaN scale":
        scales[(*at, 1)] = float("nan")
    dk, dv = (kquant.dequantize(*kquant.quantize(x)) for x in (k, v))
    got = kquant.sdpa_fa_prefill_q8(q[:, :, past:], *prefix, dk[:, :, past:], dv[:, :, past:], 256 ** -0.5).cpu().numpy()
    step = kquant.sdpa_decode_q8(q[:, :, past:past + 1].contiguous(), *prefix, 256 ** -0.5).cpu().numpy()
    hit = ~np.isfinite(step)
    assert hit[0, 4:, :, 64:128].all() and not hit[0, :4].any() and bool(hit[0, 4:].all()) == (side == "key")
    np.testing.assert_array_equal(~np.isfinite(got), np.broadcast_to(hit, got.shape))
    want = qwen.causal_prefill_attention(q[:, :, past:].cpu().numpy(), dk.cpu().numpy(), dv.cpu().numpy(), 256 ** -0.5, past=past)
    assert np.abs(np.where(np.isfinite(got), got - want, 0.0)).max() < 2e-3


@pytest.mark.parametrize("tokens", [40, 200, 1030])
@pytest.mark.parametrize("side", ["key", "value"])
def test_a_chunk_row_that_is_not_finite_reaches_the_queries_that_see_it_and_no_other(tokens, side):
    gen = torch.Generator(device="cuda").manual_seed(tokens)
    q, k, v = (torch.randn((1, h, 33 + tokens, 256), device="cuda", generator=gen).mul_(0.1) for h in (8, 2, 2))
    dk, dv = (kquant.dequantize(*kquant.quantize(x)) for x in (k, v))
    prefix = [t[:, :, :33] for t in (*kquant.quantize(k), *kquant.quantize(v))]
    want = qwen.causal_prefill_attention(q[:, :, 33:].cpu().numpy(), dk.cpu().numpy(), dv.cpu().numpy(), 256 ** -0.5, past=33)
    row = tokens // 2 + 3
    (dk if side == "key" else dv)[0, 1, 33 + row, 64:128] = float("inf") if tokens == 40 else float("nan")
    got = kquant.sdpa_fa_prefill_q8(q[:, :, 33:], *prefix, dk[:, :, 33:], dv[:, :, 33:], 256 ** -0.5).cpu().numpy()
    assert np.isnan(got[0, 4:, row:]).all()
    rest = np.abs(got - want)
    assert rest[0, :4].max() < 2e-3 and rest[0, 4:, :row].max() < 2e-3
