"""The prefill attention kernel at the edges of its tiles, head blocks and id staging, in all three forms of the dispatch."""

import numpy as np
import pytest
import torch

from oracle import ds4

pytestmark = pytest.mark.gpu


# tokens, heads, top_k, window, raw_cap, pos0, ratio: no ids; one row more or less than a tile of 32; heads of a partly
# filled wave and of a second block; the longest id list the kernel stages, and one that goes to the split kernel
@pytest.mark.parametrize("tokens,heads,top_k,window,raw_cap,pos0,ratio", [
    (1, 8, 0, 128, 1, 0, 4), (3, 16, 1, 1, 3, 9, 4), (5, 24, 31, 31, 40, 200, 4), (4, 64, 32, 32, 36, 300, 1),
    (2, 72, 33, 33, 37, 400, 4), (2, 136, 65, 128, 130, 1000, 4), (2, 16, 3520, 64, 70, 20000, 4), (2, 16, 3521, 64, 70, 20000, 4),
    (6, 32, 100, 0, 6, 0, 0)])
@pytest.mark.parametrize("form", [None, "1", "0"])
def test_edges_match_the_oracle(monkeypatch, form, tokens, heads, top_k, window, raw_cap, pos0, ratio):
    from moespresso_amd.runtime.deepseek_v4 import indexed_attention_kernel as iak

    monkeypatch.delenv("MSPR_PREFILL_PERSISTENT", raising=False)
    if form is not None:
        monkeypatch.setenv("MSPR_PREFILL_PERSISTENT", form)
    rng = np.random.default_rng(17)
    n_comp = max(8, top_k + 9)
    q = rng.standard_normal((tokens, heads, 512), dtype=np.float32)
    raw = rng.standard_normal((raw_cap, 512), dtype=np.float32).astype(np.float16)
    comp = rng.standard_normal((n_comp, 512), dtype=np.float32).astype(np.float16)
    ids = np.stack([np.sort(rng.choice(n_comp, top_k, replace=False)) for _ in range(tokens)]).astype(np.int32).reshape(tokens, top_k)
    ids[rng.random(ids.shape) < 0.1] = -1
    sinks = rng.standard_normal((heads,), dtype=np.float32)
    raw_start = raw_cap // 3
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    got = iak.indexed_mixed_attention_prefill(to(q), to(raw), to(comp), to(ids), to(sinks), pos0=pos0, window=window, ratio=ratio,
                                              raw_start=raw_start)
    want = ds4.indexed_mixed_attention_prefill(q, raw, comp, ids, sinks, pos0=pos0, window=window, ratio=ratio,
                                               raw_start=raw_start)
    np.testing.assert_allclose(got.cpu().numpy(), want, rtol=2e-3, atol=2e-3)


# a part-filled last round of workgroups in key ranges: alone, behind a whole round, in two head blocks, ids that end early,
# tokens whose last ranges hold nothing, more tokens than are worth cutting at a short list
@pytest.mark.parametrize("batch,tokens,heads,top_k,pos0", [(1, 1, 64, 512, 3000), (1, 20, 64, 512, 0), (1, 515, 16, 130, 900),
                                                          (2, 7, 72, 300, 500), (1, 80, 32, 512, 2100), (1, 81, 32, 512, 2100)])
def test_last_round_in_key_ranges(monkeypatch, batch, tokens, heads, top_k, pos0):
    from moespresso_amd.runtime.deepseek_v4 import indexed_attention_kernel as iak

    gen = torch.Generator(device="cuda").manual_seed(tokens)
    q = torch.randn((batch, heads, tokens, 512), device="cuda", generator=gen)
    raw = torch.randn((batch, 1, min(127, pos0) + tokens, 512), device="cuda", generator=gen).half()
    comp = torch.randn((batch, 900, 512), device="cuda", generator=gen).half()
    ids = torch.rand((batch, tokens, 900), device="cuda", generator=gen).topk(top_k, dim=2).indices.sort(dim=2).values.to(torch.int32)
    sinks = torch.randn(heads, device="cuda", generator=gen)
    run = lambda: iak.indexed_mixed_attention_prefill_live_f32(q, raw, comp, ids, sinks, pos0=pos0, window=128, ratio=4)
    monkeypatch.delenv("MSPR_PREFILL_PERSISTENT", raising=False)
    got = run()
    for b in range(batch):
        want = ds4.indexed_mixed_attention_prefill(q[b].transpose(0, 1).cpu().numpy(), raw[b, 0].cpu().numpy(), comp[b].cpu().numpy(),
                                                   ids[b].cpu().numpy(), sinks.cpu().numpy(), pos0=pos0, window=128, ratio=4)
        np.testing.assert_allclose(got[b].transpose(0, 1).cpu().numpy(), want, rtol=2e-3, atol=2e-3)
    monkeypatch.setenv("MSPR_PREFILL_PERSISTENT", "1")
    torch.testing.assert_close(got, run(), rtol=2e-3, atol=2e-3)


# cut rounds: three ranges (the most of them that leave one workgroup to a CU) and one token more, eight ranges, two sequences of
# two head blocks, behind a whole round, a wide ring; each with ids of which most are not visible yet: ranges that end early or
# hold nothing
@pytest.mark.parametrize("batch,tokens,heads,top_k,pos0,window", [
    (1, 85, 32, 512, 3000, 128), (1, 86, 32, 512, 3000, 128), (1, 5, 64, 1024, 3500, 128), (2, 7, 72, 300, 2000, 128),
    (1, 560, 8, 400, 2400, 64), (1, 9, 40, 256, 3000, 600)])
@pytest.mark.parametrize("first_id", [0, 500])
def test_cut_rounds_match_the_oracle(batch, tokens, heads, top_k, pos0, window, first_id):
    from moespresso_amd.runtime.deepseek_v4 import indexed_attention_kernel as iak

    gen = torch.Generator(device="cuda").manual_seed(tokens + first_id)
    q = torch.randn((batch, heads, tokens, 512), device="cuda", generator=gen).half()
    raw = torch.randn((batch, 1, window - 1 + tokens, 512), device="cuda", generator=gen).half()
    comp = torch.randn((batch, 1600, 512), device="cuda", generator=gen).half()
    ids = first_id + torch.rand((batch, tokens, 1600 - first_id), device="cuda", generator=gen).topk(top_k, dim=2).indices.sort(dim=2).values
    sinks = torch.randn(heads, device="cuda", generator=gen)
    got = iak.indexed_mixed_attention_prefill_live_f16(q, raw, comp, ids.to(torch.int32), sinks, pos0=pos0, window=window, ratio=4)
    for b in range(batch):
        want = ds4.indexed_mixed_attention_prefill(q[b].transpose(0, 1).float().cpu().numpy(), raw[b, 0].cpu().numpy(),
                                                   comp[b].cpu().numpy(), ids[b].cpu().numpy(), sinks.cpu().numpy(), pos0=pos0,
                                                   window=window, ratio=4)
        np.testing.assert_allclose(got[b].transpose(0, 1).cpu().numpy(), want, rtol=2e-3, atol=2e-3)


def test_scratch_for_fewer_ranges_cuts_into_fewer():
    from moespresso_amd import _lib

    gen = torch.Generator(device="cuda").manual_seed(6)
    tokens, n_ids, pool, pos0 = 16, 512, 900, 3600
    q = torch.randn((1, 64, tokens, 512), device="cuda", generator=gen).half()
    raw = torch.randn((1, 1, 127 + tokens, 512), device="cuda", generator=gen).half()
    comp = torch.randn((1, pool, 512), device="cuda", generator=gen).half()
    ids = torch.rand((1, tokens, pool), device="cuda", generator=gen).topk(n_ids, dim=2).indices.sort(dim=2).values.to(torch.int32)
    sinks = torch.randn(64, device="cuda", generator=gen)
    want = ds4.indexed_mixed_attention_prefill(q[0].transpose(0, 1).float().cpu().numpy(), raw[0, 0].cpu().numpy(), comp[0].cpu().numpy(),
                                               ids[0].cpu().numpy(), sinks.cpu().numpy(), pos0=pos0, window=128, ratio=4)
    part = 64 * 514 * 4
    full = _lib.lib().mspr_indexed_mixed_attention_prefill_workspace_bytes(1, 1, 64, tokens, 128, n_ids)
    assert full == 8 * tokens * part
    for nbytes in (full, 3 * tokens * part + 16, 2 * tokens * part, 2 * tokens * part - 4, 0):
        ws = torch.empty(max(nbytes, 4) // 4, device="cuda")
        out = torch.full_like(q, float("nan"), dtype=torch.float32)
        _lib.check(_lib.lib().mspr_indexed_mixed_attention_prefill(
            _lib.ptr(q), 1, 1, 64, tokens, 64 * tokens * 512, tokens * 512, 512, _lib.ptr(raw), 127 + tokens, _lib.ptr(comp), pool,
            _lib.ptr(ids), n_ids, _lib.ptr(sinks), pos0, 128, 4, 0, _lib.ptr(out), _lib.ptr(ws) if nbytes else None, nbytes,
            _lib.stream_ptr()), "prefill")
        np.testing.assert_allclose(out[0].transpose(0, 1).cpu().numpy(), want, rtol=2e-3, atol=2e-3)
