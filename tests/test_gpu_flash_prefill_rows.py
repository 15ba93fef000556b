"""GPU: query rows in and output rows out of the flash prefill kernel, element by element.

Key j of the prefix is 64 times the unit vector of column j % 256 and a query is 64 times the unit vector of its own
column, so with scale 1/16 one residue of keys scores 256 and every other key 0: the others' weights, exp(-256), are zero in
float32 and the output is the mean of that residue's value rows. The value rows are equal within a residue and hold
whole numbers from 0 to 255, which every 16-bit type, the 8-bit codes (scale 1, bias 0) and the sums over a residue hold
exactly; float32 means are taken over powers of two. A row, column or head that went to another place therefore shows, and the comparison is exact.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(Hq, Hkv, L, past, seed):
    g = torch.Generator().manual_seed(seed)
    j = torch.arange(past) % 256
    k = torch.zeros((1, Hkv, past, 256))
    k[:, :, torch.arange(past), j] = 64.0
    rows = torch.randint(0, 256, (1, Hkv, 256, 256), generator=g).float()
    rows[..., ::64], rows[..., 1::64] = 0.0, 255.0  # every group of 64 spans the codes
    v = rows[:, :, j]
    col = torch.randint(0, 256, (1, Hq, L), generator=g)
    q = torch.zeros((1, Hq, L, 256)).scatter_(3, col[..., None], 64.0)
    want = torch.stack([rows[0, h // (Hq // Hkv), col[0, h]] for h in range(Hq)])[None]
    return q, k, v, want


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Hq,Hkv,L,past", [
    (16, 2, 1, 256), (16, 2, 31, 512), (16, 2, 32, 2048), (16, 2, 97, 768), (16, 2, 203, 2048), (16, 2, 1600, 256),
    (8, 2, 33, 512), (8, 2, 161, 768), (4, 2, 130, 512), (2, 2, 64, 256), (2, 2, 300, 1024), (2, 1, 1, 256),
    (16, 4, 350, 8192), (8, 2, 333, 16384), (16, 2, 290, 256), (6, 3, 450, 8192),  # long ranges; ranges without keys
])
def test_rows_of_dense_prefill(Hq, Hkv, L, past, dtype):
    from moespresso_amd.runtime.qwen import kquant

    q, k, v, want = _case(Hq, Hkv, L, past, seed=L + past)
    tail = torch.zeros((1, Hkv, L, 256))
    dev = torch.device("cuda:0")
    got = kquant.flash_prefill(q.to(dev, dtype), torch.cat([k, tail], 2).to(dev, dtype),
                               torch.cat([v, tail], 2).to(dev, dtype), 0.0625, past_len=past)
    assert torch.equal(got.cpu().float(), want)


@pytest.mark.parametrize("sb_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("Hq,Hkv,L,past", [
    (16, 2, 1, 256), (16, 2, 33, 2048), (16, 2, 97, 512), (16, 2, 160, 32768), (16, 2, 203, 2048), (16, 4, 320, 2048),
    (8, 2, 129, 4096), (4, 2, 256, 8192), (2, 2, 48, 1024), (16, 2, 1025, 256),
    (16, 2, 500, 8192), (16, 2, 128, 32768),
])
def test_rows_of_quantised_prefill(Hq, Hkv, L, past, sb_dtype):
    from moespresso_amd.runtime.qwen import kquant

    q, k, v, want = _case(Hq, Hkv, L, past, seed=L + past)
    dev = torch.device("cuda:0")

    def codes(x):
        return x.to(torch.uint8).contiguous().view(torch.int32).view(torch.uint32).to(dev)

    one, zero = (torch.full((1, Hkv, past, 4), c, dtype=sb_dtype, device=dev) for c in (1.0, 0.0))
    chunk = torch.zeros((1, Hkv, L, 256), device=dev)
    got = kquant.sdpa_fa_prefill_q8(q.to(dev), codes(k), one, zero, codes(v), one, zero, chunk, chunk, 0.0625)
    assert torch.equal(got.cpu(), want)


@pytest.mark.parametrize("L,past", [(1, 256), (97, 512), (203, 2048), (128, 32768), (1025, 256)])
def test_quantised_prefill_may_overwrite_its_queries(L, past):
    """Rounded queries lie in the output until the merge writes it, unless that is where the queries themselves are."""
    from moespresso_amd import _lib

    q, k, v, want = _case(16, 2, L, past, seed=L + past)
    dev = torch.device("cuda:0")
    kw, vw = (x.to(torch.uint8).contiguous().to(dev) for x in (k, v))
    one, zero = (torch.full((1, 2, past, 4), c, device=dev) for c in (1.0, 0.0))
    chunk = torch.zeros((1, 2, L, 256), device=dev)
    ws = torch.empty(int(_lib.lib().mspr_sdpa_fa_prefill_q8_workspace_bytes(1, 16, 2, L, past)), dtype=torch.uint8, device=dev)
    for shared in (False, True):
        queries = q.to(dev)
        out = queries if shared else torch.full_like(queries, float("nan"))
        _lib.check(_lib.launch(
            dev, "mspr_sdpa_fa_prefill_q8",
            _lib.ptr(queries), _lib.ptr(kw), _lib.ptr(one), _lib.ptr(zero), _lib.ptr(vw), _lib.ptr(one), _lib.ptr(zero), 0,
            _lib.ptr(chunk), _lib.ptr(chunk), 0, 1, 16, 2, 256, L, past, past, 0.0625, 64, 8, _lib.ptr(out), _lib.ptr(ws),
            ws.numel()), "sdpa_fa_prefill_q8")
        assert torch.equal(out.cpu(), want), shared
        if not shared:
            assert torch.equal(queries.cpu(), q)


@pytest.mark.parametrize("name", ["queries", "k_codes", "k_scales", "k_biases", "v_codes", "v_scales", "v_biases", "chunk_k", "chunk_v"])
@pytest.mark.parametrize("L,past", [(97, 512), (97, 2048), (203, 2048)])  # prefix unpacked in the kernel, and converted
def test_quantised_prefill_may_overwrite_any_operand(L, past, name):
    """With four key ranges or more the output is written by the merge alone, when every operand has been read: it may overlap
    any of them, the whole or an end of it. (Rounded queries must then not wait in it.)"""
    from moespresso_amd import _lib

    lib, dev = _lib.lib(), torch.device("cuda:0")
    out_bytes = 16 * L * 256 * 4
    # a range's partials: a row of float32 sums and two numbers for each query of a head
    assert lib.mspr_flash_prefill_workspace_bytes(1, 16, 2, L, past) >= 4 * (out_bytes + 16 * L * 8)
    q, k, v, want = _case(16, 2, L, past, seed=L + past)
    one, zero, chunk = torch.ones((1, 2, past, 4)), torch.zeros((1, 2, past, 4)), torch.zeros((1, 2, L, 256))
    host = dict(queries=q, k_codes=k.to(torch.uint8), k_scales=one, k_biases=zero, v_codes=v.to(torch.uint8), v_scales=one,
                v_biases=zero, chunk_k=chunk, chunk_v=chunk)
    ws = torch.empty(int(lib.mspr_sdpa_fa_prefill_q8_workspace_bytes(1, 16, 2, L, past)), dtype=torch.uint8, device=dev)
    raw = host[name].contiguous().view(torch.uint8).reshape(-1)
    half = raw.numel() // 32 * 16
    for shift in (0, half, raw.numel() - 16, 16 - out_bytes, half - out_bytes):     # of the output against the operand
        ops = {n: t.to(dev) for n, t in host.items()}
        arena = torch.full((out_bytes * 2 + raw.numel() + 64,), 0xFF, dtype=torch.uint8, device=dev)
        at = out_bytes + 16                              # (the arena starts at a multiple of 256, so both are multiples of 16)
        arena[at:at + raw.numel()] = raw.to(dev)
        ops[name] = arena[at:at + raw.numel()]
        out = arena[at + shift:at + shift + out_bytes]
        p = {n: _lib.ptr(t) for n, t in ops.items()}
        _lib.check(_lib.launch(
            dev, "mspr_sdpa_fa_prefill_q8",
            p["queries"], p["k_codes"], p["k_scales"], p["k_biases"], p["v_codes"], p["v_scales"], p["v_biases"], 0,
            p["chunk_k"], p["chunk_v"], 0, 1, 16, 2, 256, L, past, past, 0.0625, 64, 8, _lib.ptr(out), _lib.ptr(ws),
            ws.numel()), "sdpa_fa_prefill_q8")
        assert torch.equal(out.view(torch.float32).reshape(want.shape).cpu(), want), shift
