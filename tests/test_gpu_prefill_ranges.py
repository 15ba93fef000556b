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


# Both sides of the line between unpacking in the attention kernel and converting beforehand: for four, three, one and two
# workgroups to a tile; behind 16384 rows (unpacked in packed arithmetic beyond); 1023 and 1024 tokens of one query head to a KV
# head (unpacked, and converted to bfloat16)
@pytest.mark.parametrize("heads,kv_heads,tokens,past", [
    (8, 2, 200, 12288), (8, 2, 200, 12289), (8, 4, 257, 3456), (8, 4, 257, 3457), (2, 2, 130, 768), (2, 2, 130, 769),
    (4, 2, 150, 3072), (4, 2, 150, 3073), (4, 1, 200, 16384), (4, 1, 200, 16385), (3, 3, 1023, 6000), (3, 3, 1024, 6000)])
def test_quantised_prefix_at_the_line_between_unpacking_and_conversion(heads, kv_heads, tokens, past):
    gen = torch.Generator(device="cuda").manual_seed(past)
    q, k, v = (torch.randn((1, h, past + tokens, 256), device="cuda", generator=gen).mul_(0.1) for h in (heads, kv_heads, kv_heads))
    tk, tv = kquant.quantize(k), kquant.quantize(v)
    dk, dv = kquant.dequantize(*tk), kquant.dequantize(*tv)
    prefix = [t[:, :, :past] for t in (*tk, *tv)]
    got = kquant.sdpa_fa_prefill_q8(q[:, :, past:], *prefix, dk[:, :, past:], dv[:, :, past:], 256 ** -0.5)
    want = qwen.causal_prefill_attention(q[:, :, past:].cpu().numpy(), dk.cpu().numpy(), dv.cpu().numpy(), 256 ** -0.5, past=past)
    assert np.abs(got.cpu().numpy() - want).max() < 2e-3


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("offset", [0.0, 3.0])
def test_unpacked_and_converted_prefixes_hold_the_same_values(dtype, offset):
    """One sequence of 700 rows is converted, two are unpacked, with the same outputs. (Scales and biases of float32 do not go
    through float16 on the way: with the offset that would move every value by up to 2^-10.)"""
    gen = torch.Generator(device="cuda").manual_seed(3)
    tokens, past = 130, 700
    q = torch.randn((1, 2, tokens, 256), device="cuda", generator=gen)
    k, v = (torch.randn((1, 2, past + tokens, 256), device="cuda", generator=gen).mul_(0.1).add_(offset).to(dtype) for _ in range(2))
    tk, tv = kquant.quantize(k), kquant.quantize(v)
    dk, dv = kquant.dequantize(*tk), kquant.dequantize(*tv)
    outs = []
    for batch in (1, 2):
        wide = lambda t: t.expand(batch, *t.shape[1:]).contiguous()
        prefix = [t[:, :, :past].view(torch.int32) if t.dtype == torch.uint32 else t[:, :, :past] for t in (*tk, *tv)]
        prefix = [wide(t) for t in prefix]
        outs.append(kquant.sdpa_fa_prefill_q8(wide(q), *prefix, wide(dk[:, :, past:]), wide(dv[:, :, past:]), 256 ** -0.5))
    assert outs[1][0].equal(outs[1][1]) and outs[1][0].equal(outs[0][0])
    want = qwen.causal_prefill_attention(q.cpu().numpy(), dk.float().cpu().numpy(), dv.float().cpu().numpy(), 256 ** -0.5, past=past)
    assert np.abs(outs[1][:1].cpu().numpy() - want).max() < 2e-3


# finite values beyond float16 saturate where the prefix is unpacked for a long chunk, as they do where it is converted
def test_unpacked_values_beyond_float16_saturate():
    gen = torch.Generator(device="cuda").manual_seed(4)
    tokens, past = 140, 2000
    q, k, v = (torch.randn((1, 2, past + tokens, 256), device="cuda", generator=gen).mul_(0.1) for _ in range(3))
    v[0, 1, 900, 70] = 3.0e5
    prefix = [t[:, :, :past] for t in (*kquant.quantize(k), *kquant.quantize(v))]
    dk, dv = (kquant.dequantize(*kquant.quantize(x)) for x in (k, v))
    got = kquant.sdpa_fa_prefill_q8(q[:, :, past:], *prefix, dk[:, :, past:], dv[:, :, past:], 256 ** -0.5).cpu().numpy()
    want = qwen.causal_prefill_attention(q[:, :, past:].cpu().numpy(), dk.cpu().numpy(), dv.clamp(-65504.0, 65504.0).cpu().numpy(),
                                         256 ** -0.5, past=past)
    assert np.isfinite(got).all()
    # (the group's other values carry the bias's float32 rounding of 3e5 / 255 steps; 2^-10 of a value for the weights)
    assert (np.abs(got - want) <= 2e-3 + 2.0 ** -9 * np.abs(want)).all()


# unpacked in the attention kernel; converted to float16; to bfloat16: one key range, several, and merges of two waves a row
@pytest.mark.parametrize("tokens,past", [(17, 40), (17, 5000), (203, 301), (203, 14000), (300, 9000), (1024, 70)])
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
