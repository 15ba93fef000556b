"""The 8-bit decode's KV heads: how far apart they lie (any distance at all for a single one), and as many as a grid takes."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,heads,n_keys,kv_rows", [(1, 1, 77, 77), (1, 1, 77, 1 << 50), (1, 2, 300, 301), (3, 2, 129, 2000)])
def test_rows_between_heads(batch, heads, n_keys, kv_rows):
    from moespresso_amd import _lib

    gen = torch.Generator(device="cuda").manual_seed(n_keys)
    held = n_keys if batch * heads == 1 else kv_rows
    codes = [torch.randint(-127, 128, (batch, heads, held, 256), device="cuda", generator=gen).to(torch.int8) for _ in range(2)]
    scales = [(torch.rand((batch, heads, held, 8), device="cuda", generator=gen) / 50).half() for _ in range(2)]
    q = torch.randn((batch, 8 * heads, 256), device="cuda", generator=gen)

    def run(k, ks, v, vs, rows):
        need = _lib.lib().mspr_sdpa_decode_q8_workspace_bytes(batch, heads, n_keys)
        ws = torch.empty(need, dtype=torch.uint8, device="cuda")
        out = torch.empty_like(q)
        _lib.check(_lib.lib().mspr_sdpa_decode_q8_0(
            _lib.ptr(q), _lib.DTYPE_CODE[q.dtype], _lib.ptr(k), _lib.ptr(ks), _lib.ptr(v), _lib.ptr(vs), batch, 8 * heads, heads, 256,
            n_keys, rows, 256 ** -0.5, _lib.ptr(out), _lib.ptr(ws), need, _lib.stream_ptr()), "q8_0")
        return out

    got = run(codes[0], scales[0], codes[1], scales[1], kv_rows)
    dense = [t[:, :, :n_keys].contiguous() for t in (codes[0], scales[0], codes[1], scales[1])]
    assert torch.equal(got, run(*dense, n_keys))


# 65536 KV heads of two sequences: the number is a word of its own among the kernel's arguments. Of 64 sequences: more merge
# workgroups than a grid of one dimension takes threads for (85 GB, most of it the partials).
@pytest.mark.parametrize("batch", [2, 64])
def test_as_many_heads_as_a_grid_takes(batch):
    """With one key the softmax is 1, so the output is that key's value row in the cache's format."""
    from moespresso_amd import _lib

    gen = torch.Generator(device="cuda").manual_seed(5)
    heads = 65536
    codes = torch.randint(-127, 128, (batch, heads, 1, 256), device="cuda", generator=gen, dtype=torch.int8)
    scales = (torch.rand((batch, heads, 1, 8), device="cuda", generator=gen) / 50).half()
    q = torch.randn((batch, heads, 256), device="cuda", generator=gen)
    need = _lib.lib().mspr_sdpa_decode_q8_workspace_bytes(batch, heads, 1)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    out = torch.empty_like(q)
    _lib.check(_lib.lib().mspr_sdpa_decode_q8_0(
        _lib.ptr(q), _lib.DTYPE_CODE[q.dtype], _lib.ptr(codes), _lib.ptr(scales), _lib.ptr(codes), _lib.ptr(scales), batch, heads, heads,
        256, 1, 1, 256 ** -0.5, _lib.ptr(out), _lib.ptr(ws), need, _lib.stream_ptr()), "q8_0")
    del ws
    for b in range(0, batch, max(1, batch // 8)):
        want = (codes[b].half().reshape(heads, 8, 32) * scales[b].reshape(heads, 8, 1)).reshape(heads, 256)
        assert torch.equal(out[b], want.float())
    del q, out, codes
    torch.cuda.empty_cache()
