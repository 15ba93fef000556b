"""What the speed of this package is measured on: the attention work of a model served from this package, through
the callables that the model's layers call. One case is one layer's share of a step, one pass is one such step.

Seven kinds of work, after the two model families that the package serves:

* ``ds4_decode``         batched decode over an fp8-key index: scores, top-k, multi-head-latent attention
* ``ds4_token``          one-token decode of a compressed-pool layer: index-query rope, fused prep, fused attention
* ``ds4_prefill``        a prompt chunk of a compressed-pool layer: ropes, QAT, scores, top-k, attention, inverse rope
* ``qwen_decode_affine`` one token into an affine 8-bit cache (quantise on append), then GQA decode over it
* ``qwen_decode_q8_0``   GQA decode over an int8 cache with one float16 scale per 32 elements
* ``qwen_prefill_q8``    a prompt chunk against an affine 8-bit cache: round trip of the chunk, append, flash prefill
* ``flash_prefill``      a prompt chunk against a dense 16-bit cache that already holds it
"""

import math

import torch

from moespresso_amd.runtime.deepseek_v4 import attention_seam_kernel as seam
from moespresso_amd.runtime.deepseek_v4 import decode_attention_kernel as dak
from moespresso_amd.runtime.deepseek_v4 import indexed_attention_kernel as iak
from moespresso_amd.runtime.deepseek_v4 import indexer_score_kernel as isk
from moespresso_amd.runtime.qwen import kquant

HEADS, INDEX_HEADS, INDEX_DIM = 64, 64, 128          # DS4 attention and index heads
ROW_DIM, MLA_DIM, ROPE_DIM = 512, 576, 64            # DS4 cache row, latent row with its rotary part, rotary width
WINDOW, RATIO = 128, 4                               # DS4 sliding window, tokens per compressed row
Q_HEADS, KV_HEADS, HEAD_DIM = 16, 2, 256             # Qwen full attention
Q8_ROW = HEAD_DIM + HEAD_DIM // 32 * 2               # bytes of an 8-bit cache row with its scales (both formats)
DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
SIZE = {"float32": 4, "float16": 2, "bfloat16": 2}


def listed():
    return [
        # one sequence of a chat at 32K tokens: three small launches' worth of work, call overhead counts
        dict(name="ds4_decode_1x8192", kind="ds4_decode", batch=1, keys=8192, topk=2048, dtype="bfloat16", sinks=False,
             layers=0),
        # a small batch at an odd context, float16 cache with sinks, called layer by layer
        dict(name="ds4_decode_5x19211", kind="ds4_decode", batch=5, keys=19211, topk=1024, dtype="float16", sinks=True,
             layers=0),
        # the served batch at 128K tokens: a decode step's layers replayed from one captured graph
        dict(name="ds4_decode_16x32768_graph", kind="ds4_decode", batch=16, keys=32768, topk=2048, dtype="bfloat16",
             sinks=False, layers=4),
        # a single user's next token after a 3844-token prompt, the smallest call of the package
        dict(name="ds4_token_961", kind="ds4_token", rows=961, topk=512, dtype="float16"),
        # the prompt itself, and a chunk of the same size deep in a long context with float32 activations
        dict(name="ds4_prefill_3844_at_0", kind="ds4_prefill", tokens=3844, pos0=0, topk=512, dtype="float16"),
        dict(name="ds4_prefill_3844_at_28000", kind="ds4_prefill", tokens=3844, pos0=28000, topk=512, dtype="float32"),
        # a follow-up turn: a short ragged chunk behind 7698 tokens
        dict(name="ds4_prefill_517_at_7698", kind="ds4_prefill", tokens=517, pos0=7698, topk=512, dtype="float16"),
        # one token of a single user at 8K tokens, quantised on append
        dict(name="qwen_decode_1x8191", kind="qwen_decode_affine", batch=1, keys=8191, dtype="bfloat16"),
        # a batch of eight at 37000 tokens
        dict(name="qwen_decode_8x37000", kind="qwen_decode_q8_0", batch=8, keys=37000, dtype="bfloat16"),
        # a follow-up turn's short chunk, and a long prompt's last 2048-token chunk
        dict(name="qwen_prefill_203_at_9001", kind="qwen_prefill_q8", tokens=203, past=9001, dtype="float32"),
        dict(name="qwen_prefill_2048_at_34952", kind="qwen_prefill_q8", tokens=2048, past=34952, dtype="bfloat16"),
        # a 4096-token chunk behind a 32768-token dense prefix
        dict(name="flash_prefill_4096_at_32768", kind="flash_prefill", tokens=4096, past=32768, dtype="bfloat16"),
    ]


def _spread(rng, low, high):
    """A whole number in [low, high], even over the logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(["ds4_decode", "ds4_decode", "ds4_token", "ds4_prefill", "ds4_prefill", "qwen_decode_affine",
                       "qwen_decode_q8_0", "qwen_prefill_q8", "flash_prefill"])
    if kind == "ds4_decode":
        layers = rng.choice([0, 0, 2, 4])
        return dict(kind=kind, batch=_spread(rng, 1, 16), keys=_spread(rng, 2100, 32768),
                    topk=rng.choice([512, 1024, 2048]), dtype=rng.choice(["bfloat16", "float16"]),
                    sinks=rng.choice([False, True]), layers=layers)
    if kind == "ds4_token":
        return dict(kind=kind, rows=_spread(rng, 520, 32768), topk=512, dtype=rng.choice(["float16", "float32"]))
    if kind == "ds4_prefill":
        tokens, pos0 = _spread(rng, 17, 3844), _spread(rng, 2100, 28000)
        if tokens >= 2100 and rng.random() < 0.5:    # a prompt from its start
            pos0 = 0
        return dict(kind=kind, tokens=tokens, pos0=pos0, topk=512, dtype=rng.choice(["float16", "float32"]))
    if kind in ("qwen_decode_affine", "qwen_decode_q8_0"):
        batch = rng.choice([1, 1, 2, 3, 4, 6, 8])
        return dict(kind=kind, batch=batch, keys=_spread(rng, 1024, 37000), dtype=rng.choice(["bfloat16", "float32"]))
    tokens, past = _spread(rng, 33, 4096), _spread(rng, 256, 32768)
    dtype = rng.choice(["bfloat16", "float32"] if kind == "qwen_prefill_q8" else ["bfloat16", "float16"])
    return dict(kind=kind, tokens=tokens, past=past, dtype=dtype)


# ------------------------------------------------------------------------------------------------ inputs

def _normal(gen, *shape, dtype=torch.float32, scale=1.0):
    t = torch.randn(shape, device="cuda", dtype=dtype, generator=gen)
    return t if scale == 1.0 else t.mul_(scale)


def _inv_freq():
    return 1.0 / 10000.0 ** (torch.arange(0, ROPE_DIM, 2, device="cuda", dtype=torch.float32) / ROPE_DIM)


def _decode_layer(case, gen):
    batch, keys, dtype = case["batch"], case["keys"], DTYPES[case["dtype"]]
    rows = _normal(gen, batch, keys, INDEX_DIM)
    key_scales = (rows.abs().amax(dim=-1) / 448.0).contiguous()
    return dict(
        q_idx=_normal(gen, batch, INDEX_HEADS, INDEX_DIM, dtype=torch.bfloat16),
        keys=(rows / key_scales[..., None]).to(torch.float8_e4m3fn), key_scales=key_scales,
        weights=torch.rand((batch, INDEX_HEADS), device="cuda", generator=gen),
        q=_normal(gen, batch, HEADS, MLA_DIM, dtype=dtype),
        kv=_normal(gen, batch, RATIO * keys, MLA_DIM, dtype=dtype),
        sinks=_normal(gen, HEADS) if case["sinks"] else None)


def _decode_layer_pass(case, s):
    scores = isk.indexer_scores_fp8(s["q_idx"], s["keys"], s["key_scales"], s["weights"])
    sel = isk.topk_select(scores, case["topk"])
    # a selected entry stands for the last of its RATIO tokens
    out = iak.sparse_mla_decode(s["q"], s["kv"], sel, scale=MLA_DIM ** -0.5,
                                window_start=RATIO * case["keys"] - WINDOW, window_rows=WINDOW, sinks=s["sinks"],
                                row_mul=RATIO, row_add=RATIO - 1)
    return {"sel": sel, "out": out}


def _prepare_ds4_decode(case, gen):
    if not case["layers"]:
        return _decode_layer(case, gen)
    layers = [_decode_layer(case, gen) for _ in range(case["layers"])]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _decode_layer_pass(case, layers[0])
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = [_decode_layer_pass(case, s) for s in layers]
    return dict(layers=layers, graph=graph, outs=outs)


def _run_ds4_decode(case, s):
    if case["layers"]:
        s["graph"].replay()
        return s["outs"]
    return _decode_layer_pass(case, s)


def _prepare_ds4_token(case, gen):
    rows, dtype = case["rows"], DTYPES[case["dtype"]]
    position = RATIO * rows + 1
    return dict(
        position=position, inv_freq=_inv_freq(),
        params=torch.tensor([position, position % WINDOW], dtype=torch.int32, device="cuda"),
        q_idx=_normal(gen, 1, INDEX_HEADS, 1, INDEX_DIM, dtype=dtype),
        pooled_qat=isk.indexer_qat_rows(_normal(gen, rows, INDEX_DIM, dtype=torch.float16)),
        weights=torch.rand((INDEX_HEADS,), device="cuda", generator=gen) * INDEX_HEADS ** -0.5,
        kv_row=_normal(gen, ROW_DIM, dtype=torch.float16), q=_normal(gen, HEADS, ROW_DIM, dtype=torch.float16),
        window=_normal(gen, WINDOW, ROW_DIM, dtype=torch.float16),
        pooled=_normal(gen, rows, ROW_DIM, dtype=torch.float16), sinks=_normal(gen, HEADS, dtype=torch.float16))


def _run_ds4_token(case, s):
    q_idx = seam.fused_partial_rope(s["q_idx"], s["inv_freq"], offset=s["position"])
    sel, row, _ = dak.fused_decode_prep(q_idx.reshape(INDEX_HEADS, INDEX_DIM), s["pooled_qat"], s["weights"],
                                        s["kv_row"], s["inv_freq"], s["params"], scale=INDEX_DIM ** -0.5,
                                        topk=case["topk"])
    heads = dak.fused_decode_sdpa(s["q"], s["window"], row, s["pooled"], sel, s["sinks"], s["inv_freq"], s["params"],
                                  scale=ROW_DIM ** -0.5)
    return {"sel": sel, "row": row, "heads": heads}


def _prepare_ds4_prefill(case, gen):
    tokens, dtype = case["tokens"], DTYPES[case["dtype"]]
    pool = (case["pos0"] + tokens) // RATIO
    return dict(
        inv_freq=_inv_freq(), q=_normal(gen, 1, HEADS, tokens, ROW_DIM, dtype=dtype),
        kv=_normal(gen, 1, 1, tokens, ROW_DIM, dtype=torch.float16),
        # ring rows of the tokens just before the chunk
        past=_normal(gen, 1, 1, min(WINDOW - 1, case["pos0"]), ROW_DIM, dtype=torch.float16),
        pooled=_normal(gen, 1, pool, ROW_DIM, dtype=torch.float16),
        q_idx=_normal(gen, 1, INDEX_HEADS, tokens, INDEX_DIM, dtype=dtype),
        pooled_qat=isk.indexer_qat_rows(_normal(gen, 1, pool, INDEX_DIM)),
        weights=torch.rand((1, tokens, INDEX_HEADS), device="cuda", generator=gen) * (INDEX_HEADS * INDEX_DIM) ** -0.5,
        sinks=_normal(gen, HEADS))


def _run_ds4_prefill(case, s):
    pos0 = case["pos0"]
    q = seam.fused_partial_rope(s["q"], s["inv_freq"], offset=pos0)
    kv = seam.fused_partial_rope(s["kv"], s["inv_freq"], offset=pos0)
    ring = torch.cat([s["past"], kv], dim=2)
    q_idx = seam.fused_partial_rope(s["q_idx"], s["inv_freq"], offset=pos0)
    q_idx = iak.indexer_q_qat_live(q_idx.to(torch.float32))
    scores = iak.indexer_scores_tiled_live(q_idx, s["weights"], s["pooled_qat"], pos0=pos0, ratio=RATIO)
    sel = isk.topk_select(scores, case["topk"])
    attend = (iak.indexed_mixed_attention_prefill_live_f16 if q.dtype == torch.float16 else
              iak.indexed_mixed_attention_prefill_live_f32)
    heads = attend(q, ring, s["pooled"], sel, s["sinks"], pos0=pos0, window=WINDOW, ratio=RATIO)
    heads = seam.fused_partial_rope(heads, s["inv_freq"], offset=pos0, inverse=True)
    return {"ring": ring, "sel": sel, "heads": heads}


def _filled_cache(gen, batch, keys, dtype):
    cache = kquant.QuantizedKVCache()
    cache.update_and_fetch(_normal(gen, batch, KV_HEADS, keys, HEAD_DIM, dtype=dtype),
                           _normal(gen, batch, KV_HEADS, keys, HEAD_DIM, dtype=dtype))
    return cache


def _words(triplet):
    """A cache triplet with its packed codes as int32, the type that every tensor operation takes."""
    return triplet[0].view(torch.int32), triplet[1], triplet[2]


def _prepare_qwen_decode_affine(case, gen):
    batch, dtype = case["batch"], DTYPES[case["dtype"]]
    return dict(cache=_filled_cache(gen, batch, case["keys"], dtype), q=_normal(gen, batch, Q_HEADS, 1, HEAD_DIM),
                k=_normal(gen, batch, KV_HEADS, 1, HEAD_DIM, dtype=dtype),
                v=_normal(gen, batch, KV_HEADS, 1, HEAD_DIM, dtype=dtype))


def _run_qwen_decode_affine(case, s):
    s["cache"].offset = case["keys"]                 # the same step again: the token goes behind the same prefix
    k, v = s["cache"].update_and_fetch(s["k"], s["v"])
    out = kquant.sdpa_decode_q8(s["q"], *k, *v, HEAD_DIM ** -0.5)
    return {"out": out, "k": _words(k), "v": _words(v)}


def _prepare_qwen_decode_q8_0(case, gen):
    batch, keys = case["batch"], case["keys"]
    cache = []
    for _ in range(2):
        x = _normal(gen, batch, KV_HEADS, keys, HEAD_DIM // 32, 32)
        scales = (x.abs().amax(dim=-1) / 127.0).to(torch.float16)
        codes = torch.round(x / scales[..., None].float()).clamp_(-127, 127).to(torch.int8)
        cache += [codes.reshape(batch, KV_HEADS, keys, HEAD_DIM), scales]
    return dict(cache=cache, q=_normal(gen, batch, Q_HEADS, HEAD_DIM, dtype=DTYPES[case["dtype"]]))


def _run_qwen_decode_q8_0(case, s):
    return kquant.sdpa_decode_q8_0(s["q"], *s["cache"], HEAD_DIM ** -0.5)


def _prepare_qwen_prefill_q8(case, gen):
    tokens, dtype = case["tokens"], DTYPES[case["dtype"]]
    return dict(cache=_filled_cache(gen, 1, case["past"], dtype), q=_normal(gen, 1, Q_HEADS, tokens, HEAD_DIM),
                k=_normal(gen, 1, KV_HEADS, tokens, HEAD_DIM, dtype=dtype),
                v=_normal(gen, 1, KV_HEADS, tokens, HEAD_DIM, dtype=dtype))


def _run_qwen_prefill_q8(case, s):
    cache = s["cache"]
    cache.offset = case["past"]                      # the same chunk again: it goes behind the same prefix
    past_k, past_v = cache.state
    self_k = kquant.dequantize(*kquant.quantize(s["k"]))
    self_v = kquant.dequantize(*kquant.quantize(s["v"]))
    k, v = cache.update_and_fetch(s["k"], s["v"])
    out = kquant.sdpa_fa_prefill_q8(s["q"], *past_k, *past_v, self_k, self_v, HEAD_DIM ** -0.5)
    return {"out": out, "k": _words(k), "v": _words(v)}


def _prepare_flash_prefill(case, gen):
    tokens, rows, dtype = case["tokens"], case["past"] + case["tokens"], DTYPES[case["dtype"]]
    return dict(q=_normal(gen, 1, Q_HEADS, tokens, HEAD_DIM, dtype=dtype, scale=0.5),
                k=_normal(gen, 1, KV_HEADS, rows, HEAD_DIM, dtype=dtype, scale=0.5),
                v=_normal(gen, 1, KV_HEADS, rows, HEAD_DIM, dtype=dtype, scale=0.5))


def _run_flash_prefill(case, s):
    return kquant.flash_prefill(s["q"], s["k"], s["v"], HEAD_DIM ** -0.5, past_len=case["past"])


_PREPARE = {"ds4_decode": _prepare_ds4_decode, "ds4_token": _prepare_ds4_token, "ds4_prefill": _prepare_ds4_prefill,
            "qwen_decode_affine": _prepare_qwen_decode_affine, "qwen_decode_q8_0": _prepare_qwen_decode_q8_0,
            "qwen_prefill_q8": _prepare_qwen_prefill_q8, "flash_prefill": _prepare_flash_prefill}
_RUN = {"ds4_decode": _run_ds4_decode, "ds4_token": _run_ds4_token, "ds4_prefill": _run_ds4_prefill,
        "qwen_decode_affine": _run_qwen_decode_affine, "qwen_decode_q8_0": _run_qwen_decode_q8_0,
        "qwen_prefill_q8": _run_qwen_prefill_q8, "flash_prefill": _run_flash_prefill}


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return case, _PREPARE[case["kind"]](case, gen)


def run(state):
    case, s = state
    return _RUN[case["kind"]](case, s)


# ------------------------------------------------------------------------------------------------ work, tolerance

def _seen(tokens, pos0, cap, ratio=1):
    """Rows that the tokens of a chunk see together: of each, those up to its own position, at most ``cap``."""
    return sum(min(cap, (pos0 + t + 1) // ratio) for t in range(tokens))


def work(case):
    kind, size = case["kind"], SIZE[case["dtype"]]
    if kind == "ds4_decode":
        rows = min(case["topk"], case["keys"]) + WINDOW
        nbytes = (case["keys"] * (INDEX_DIM + 4) + INDEX_HEADS * (INDEX_DIM * 2 + 4) + case["topk"] * 4
                  + rows * MLA_DIM * size + HEADS * (MLA_DIM + ROW_DIM) * size)
        flops = 2 * INDEX_HEADS * INDEX_DIM * case["keys"] + 2 * HEADS * (MLA_DIM + ROW_DIM) * rows
        times = case["batch"] * max(1, case["layers"])
        return {"bytes": times * nbytes, "flops": times * flops}
    if kind == "ds4_token":
        rows = case["topk"] + WINDOW
        return {"bytes": (case["rows"] * INDEX_DIM * 4 + INDEX_HEADS * (INDEX_DIM * size + 4) + case["topk"] * 4
                          + rows * ROW_DIM * 2 + (2 * HEADS + 2) * ROW_DIM * 2),
                "flops": 2 * INDEX_HEADS * INDEX_DIM * case["rows"] + 4 * HEADS * ROW_DIM * rows}
    if kind == "ds4_prefill":
        tokens, pos0 = case["tokens"], case["pos0"]
        pool = (pos0 + tokens) // RATIO
        seen = _seen(tokens, pos0, WINDOW) + _seen(tokens, pos0, min(case["topk"], pool), RATIO)
        return {"bytes": (tokens * (HEADS * ROW_DIM * (size + 4) + INDEX_HEADS * (INDEX_DIM * size + 4))
                          + tokens * (2 * ROW_DIM * 2 + case["topk"] * 4) + 2 * min(WINDOW - 1, pos0) * ROW_DIM * 2
                          + pool * (ROW_DIM * 2 + INDEX_DIM * 4)),
                "flops": (2 * INDEX_HEADS * INDEX_DIM * _seen(tokens, pos0, pool, RATIO)
                          + 4 * HEADS * ROW_DIM * seen)}
    if kind in ("qwen_decode_affine", "qwen_decode_q8_0"):
        keys = case["keys"] + (kind == "qwen_decode_affine")
        row = Q8_ROW if kind == "qwen_decode_q8_0" else HEAD_DIM + HEAD_DIM // 64 * 2 * size
        io = 2 * size if kind == "qwen_decode_q8_0" else 2 * 4
        return {"bytes": case["batch"] * (2 * KV_HEADS * keys * row + Q_HEADS * HEAD_DIM * io),
                "flops": case["batch"] * 4 * Q_HEADS * HEAD_DIM * keys}
    tokens, past = case["tokens"], case["past"]
    flops = 4 * Q_HEADS * HEAD_DIM * _seen(tokens, past, past + tokens)
    if kind == "qwen_prefill_q8":
        row = HEAD_DIM + HEAD_DIM // 64 * 2 * size
        return {"bytes": (2 * KV_HEADS * (past * row + tokens * (HEAD_DIM * size + row))
                          + 2 * Q_HEADS * tokens * HEAD_DIM * 4), "flops": flops}
    return {"bytes": 2 * (KV_HEADS * (past + tokens) + Q_HEADS * tokens) * HEAD_DIM * size, "flops": flops}


def tolerance(case):
    """Selections, cache codes and cache rows are exact but for selections whose scores tie within the rounding of
    their sums; attention follows the type its weights are rounded to (bfloat16 or float16)."""
    kind = case["kind"]
    differ = 0.01 if kind.startswith("ds4") else 0.0
    half = kind in ("ds4_token", "ds4_prefill", "qwen_decode_affine", "qwen_decode_q8_0") or case["dtype"] == "float16"
    if kind == "qwen_decode_q8_0" and case["dtype"] == "bfloat16":
        half = False                                 # the output itself is bfloat16
    return {"rel": 2e-3 if half else 1e-2, "differ": differ}
