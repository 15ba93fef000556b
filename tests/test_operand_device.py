"""Operands that live on another device than the current one (CPU: fake tensors, a recorded library)."""

import contextlib

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from moespresso_amd import _lib
from moespresso_amd.runtime.deepseek_v4 import attention_seam_kernel as seam
from moespresso_amd.runtime.deepseek_v4 import indexed_attention_kernel as iak
from moespresso_amd.runtime.deepseek_v4 import indexer_score_kernel as isk
from moespresso_amd.runtime.qwen import kquant


def _bf16(*shape):
    return torch.empty(shape, dtype=torch.bfloat16, device="cuda:1")


def _f32(*shape):
    return torch.empty(shape, device="cuda:1")


CALLS = {
    "mspr_topk_select": lambda: isk.topk_select(_f32(3, 700), 64),
    "mspr_indexer_qat_rows": lambda: isk.indexer_qat_rows(_f32(5, 128)),
    "mspr_indexer_q_qat_live": lambda: iak.indexer_q_qat_live(_f32(1, 4, 2, 128)),
    "mspr_fused_partial_rope": lambda: seam.fused_partial_rope(_f32(1, 4, 2, 512), _f32(32), offset=3),
    "mspr_sparse_mla_decode": lambda: iak.sparse_mla_decode(
        _bf16(1, 64, 576), _bf16(1, 900, 576), torch.empty((1, 40), dtype=torch.int32, device="cuda:1"), scale=0.1),
    "mspr_affine_q8_quantize": lambda: kquant.quantize(_f32(1, 2, 3, 256)),
    "mspr_flash_prefill": lambda: kquant.flash_prefill(_bf16(1, 4, 8, 256), _bf16(1, 2, 40, 256), _bf16(1, 2, 40, 256), 0.1,
                                                       past_len=32),
}


@pytest.mark.skipif(not _lib.library_available(), reason="the library is not built")
@pytest.mark.parametrize("entry", sorted(CALLS))
@pytest.mark.parametrize("current", [0, 1])
def test_a_call_is_launched_on_the_stream_of_its_operands_device(monkeypatch, entry, current):
    on = [current]
    launched = []

    @contextlib.contextmanager
    def device(d):
        on.append(d.index)
        yield
        on.pop()

    class Library:
        def __getattr__(self, name):
            if name.endswith("_bytes"):
                return getattr(real, name)
            return lambda *args: launched.append((name, on[-1], args[-1])) or 0

    real = _lib.lib()
    monkeypatch.setattr(_lib, "lib", Library)
    monkeypatch.setattr(_lib, "ptr", lambda t: None)
    monkeypatch.setattr(_lib, "stream_ptr", lambda: f"stream of {on[-1]}")
    monkeypatch.setattr(torch.cuda, "current_device", lambda: on[-1])
    monkeypatch.setattr(torch.cuda, "device", device)
    with FakeTensorMode():
        CALLS[entry]()
    assert launched == [(entry, 1, "stream of 1")] and on == [current]


@pytest.mark.skipif(isinstance(_lib.dispatch, _lib._NoNativePath), reason="the native call path is not built")
def test_the_native_path_leaves_operands_of_another_device_to_python():
    with FakeTensorMode():
        x, bf = _f32(1, 2, 3, 256), _bf16(1, 64, 576)
        rows = torch.empty((1, 40), dtype=torch.int32, device="cuda:1")
        wq = torch.empty((1, 2, 3, 64), dtype=torch.int32, device="cuda:1").view(torch.uint32)
        pool = _bf16(1, 900, 576)
        qat, inv, sb = _f32(1, 4, 2, 128), _f32(32), _f32(1, 2, 3, 4)
    native = _lib.dispatch
    assert native.topk_select(x, 8) is None
    assert native.indexer_qat_rows(qat) is None
    assert native.indexer_q_qat_live(qat) is None
    assert native.quantize(x) is None
    assert native.dequantize(wq, sb, sb) is None
    assert native.fused_partial_rope(x, inv, 3, False, None, 1 << 20) is None
    assert native.sparse_mla_decode(bf, pool, rows, 0.1, 512, None, 0, None, None, 1, 0) is None
