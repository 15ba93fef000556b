"""Which chunks have their quantised prefix converted before attention, read off the scratch that the call asks for (CPU)."""

import pytest

from moespresso_amd import _lib

pytestmark = pytest.mark.skipif(not _lib.library_available(), reason="the library is not built")


def converted(heads, kv_heads, tokens, past, batch=1):
    """True if scratch has room for 16-bit rows of the whole prefix, False if only for the rows of its last, part-filled tile."""
    lib = _lib.lib()
    need = lib.mspr_sdpa_fa_prefill_q8_workspace_bytes(batch, heads, kv_heads, tokens, past)
    partials = lib.mspr_flash_prefill_workspace_bytes(batch, heads, kv_heads, tokens, past)
    rows = (need - partials) // (batch * kv_heads * 256 * 2 * 2)
    assert rows in (past + tokens, past % 32 + tokens), rows
    return rows == past + tokens


def test_few_workgroups_to_a_tile_unpack_a_long_prefix():
    # (us unpacked and converted: 4 / 4 heads, 256 over 16000 rows 53 and 65; 16 / 4, 160 over 16000 82 and 88)
    assert not converted(4, 4, 256, 16000) and not converted(4, 4, 512, 8000) and not converted(16, 4, 160, 16000)
    assert not converted(8, 2, 160, 12000) and not converted(16, 4, 257, 32000)
    assert converted(16, 4, 160, 2000) and converted(16, 4, 512, 16000)
    assert converted(16, 2, 203, 9001) and converted(16, 2, 160, 16384) and not converted(16, 2, 160, 16385)
    assert converted(16, 2, 160, 13824, batch=2) and not converted(16, 2, 160, 13825, batch=2)
    assert converted(16, 2, 256, 16384) and not converted(16, 2, 256, 16385) and converted(16, 2, 257, 33333)


def test_short_chunks_unpack_and_long_ones_convert():
    for heads, kv_heads in ((16, 2), (8, 2), (4, 4), (2, 1)):
        for past in (33, 1000, 9001, 33333):
            assert not converted(heads, kv_heads, 128, past)
            assert converted(heads, kv_heads, 1024, past)    # (staged as bfloat16, which only the converted form reads)
