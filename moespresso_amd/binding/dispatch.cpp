// Native call path of the operators: torch tensors in, one C-ABI call, torch tensors out.
//
// At batch 1 a decode layer is a handful of kernels of 4 to 12 us, and a call made in Python (shape checks, two
// allocations, twenty converted arguments) costs the host as much as its kernels cost the device: three such calls of
// the DS4 decode layer took 42 us of host time against 30 us of kernels. Each function here takes the arguments of one
// Python operator by position, checks the plain case (types, shapes, dense layout, the current device) and makes the call.
// Whatever is not that case (another layout, a type to convert, a mistake) makes it return None, and the Python operator
// goes through its own checks, conversions and messages; so nothing is rejected or converted here.
//
// Outputs and scratch come from torch's allocator on the current stream. The interpreter lock is released around the
// launches, as it is around a foreign call made from Python.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <initializer_list>

#include "../../include/moespresso_amd.h"

namespace {

using at::Tensor;

constexpr int kNoType = -1;

int type_code(at::ScalarType t) {
  return t == at::kFloat ? MSPR_F32 : t == at::kHalf ? MSPR_F16 : t == at::kBFloat16 ? MSPR_BF16 : kNoType;
}

// The tensor an argument holds, if it is a dense one on a HIP device.
const Tensor* dense(PyObject* o, int64_t ndim) {
  if (!THPVariable_Check(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  return t.defined() && t.is_cuda() && t.dim() == ndim && t.is_contiguous() ? &t : nullptr;
}

const Tensor* dense(PyObject* o, int64_t ndim, at::ScalarType type) {
  const Tensor* t = dense(o, ndim);
  return t && t->scalar_type() == type ? t : nullptr;
}

// Launches go to the current device's stream: operands of another one are the Python path's, which changes devices.
bool here(const Tensor& t) {
  c10::DeviceIndex current;
  return t.is_cuda() && c10::hip::GetDevice(&current) == hipSuccess && t.get_device() == current;
}

bool here(std::initializer_list<const Tensor*> ts) {
  const Tensor* first = *ts.begin();
  for (const Tensor* t : ts)
    if (t->get_device() != first->get_device()) return false;
  return here(*first);
}

// Whole numbers and real numbers that are Python's own; anything else (NumPy scalars, tensors) is the Python path's.
bool whole(PyObject* o, int64_t* v) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  *v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}

bool whole32(PyObject* o, int* v) {
  int64_t w;
  if (!whole(o, &w) || w < INT32_MIN || w > INT32_MAX) return false;
  *v = (int)w;
  return true;
}

bool real(PyObject* o, float* v) {
  if (!PyFloat_CheckExact(o)) return false;
  *v = (float)PyFloat_AS_DOUBLE(o);
  return true;
}

Tensor empty(at::IntArrayRef shape, at::ScalarType type, const Tensor& like) {
  return at::detail::empty_cuda(shape, type, like.device(), std::nullopt);
}

Tensor scratch(size_t nbytes, const Tensor& like) {
  return empty({(int64_t)((nbytes < 16 ? 16 : nbytes) + 3) / 4}, at::kFloat, like);
}

void* stream() { return (void*)c10::hip::getCurrentHIPStream().stream(); }

const void* at_or_null(const Tensor* t) { return t ? t->const_data_ptr() : nullptr; }

// Scratch the caller handed over, or a new one of the size asked for. False: not a plain scratch tensor.
bool take_workspace(PyObject* o, size_t nbytes, const Tensor& like, Tensor* ws) {
  if (o == Py_None) {
    *ws = scratch(nbytes, like);
    return true;
  }
  if (!THPVariable_Check(o)) return false;
  *ws = THPVariable_Unpack(o);
  return ws->is_cuda() && ws->is_contiguous() && ws->get_device() == like.get_device();
}

PyObject* none() { Py_RETURN_NONE; }

bool failed(int rc, const char* what) {
  if (rc == MSPR_OK) return false;
  PyErr_Format(rc == MSPR_ERR_ARG ? PyExc_ValueError : PyExc_RuntimeError, "%s: %s", what, mspr_last_error());
  return true;
}

// The launches of one call, with the interpreter lock released.
template <typename F>
int launch(F&& call) {
  void* st = stream();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = call(st);
  Py_END_ALLOW_THREADS
  return rc;
}

PyObject* wrap(const Tensor& t) { return THPVariable_Wrap(t); }

template <typename... T>
PyObject* wrap_tuple(const T&... ts) {
  PyObject* r = PyTuple_New(sizeof...(ts));
  if (!r) return nullptr;
  Py_ssize_t i = 0;
  (PyTuple_SET_ITEM(r, i++, THPVariable_Wrap(ts)), ...);
  return r;
}

#define MSPR_NARGS(n)                                                                       \
  if (nargs != (n)) {                                                                       \
    PyErr_Format(PyExc_TypeError, "%s takes %d arguments, %zd given", __func__, n, nargs); \
    return nullptr;                                                                         \
  }

// Every entry point may see C++ exceptions of the allocator (out of memory): they become Python's.
template <PyObject* (*F)(PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  return F(a, nargs);
  END_HANDLE_TH_ERRORS
}

// ---------------------------------------------------------------------------------------------- DS4 indexer

// (x [..., 128]) -> float32, same shape
template <bool LIVE>
PyObject* qat_rows(PyObject* const* a, Py_ssize_t nargs) {
  MSPR_NARGS(1)
  if (!THPVariable_Check(a[0])) return none();
  const Tensor& x = THPVariable_Unpack(a[0]);
  if (!here(x) || x.dim() < 1 || x.size(-1) != 128 || x.numel() == 0 || !x.is_contiguous()) return none();
  const int code = type_code(x.scalar_type());
  if (code == kNoType || (LIVE && (code != MSPR_F32 || x.dim() != 4))) return none();
  Tensor out = empty(x.sizes(), at::kFloat, x);
  const int64_t n = x.numel() / 128;
  const int rc = launch([&](void* st) {
    return LIVE ? mspr_indexer_q_qat_live((const float*)x.const_data_ptr(), n, (float*)out.data_ptr(), st)
                : mspr_indexer_qat_rows(x.const_data_ptr(), code, n, (float*)out.data_ptr(), st);
  });
  return failed(rc, LIVE ? "indexer_q_qat_live" : "indexer_qat_rows") ? nullptr : wrap(out);
}

// (scores float32 [..., n_rows], topk) -> int32 [..., topk]
PyObject* topk_select(PyObject* const* a, Py_ssize_t nargs) {
  MSPR_NARGS(2)
  int64_t k;
  if (!THPVariable_Check(a[0]) || !whole(a[1], &k)) return none();
  const Tensor& s = THPVariable_Unpack(a[0]);
  if (!here(s) || s.dim() < 1 || s.scalar_type() != at::kFloat || !s.is_contiguous()) return none();
  const int64_t n = s.size(-1);
  if (k < 1 || k > n || s.numel() == 0) return none();
  at::DimVector shape(s.sizes());
  shape.back() = k;
  Tensor sel = empty(shape, at::kInt, s);
  const int rc = launch([&](void* st) {
    return mspr_topk_select((const float*)s.const_data_ptr(), n, (int)(s.numel() / n), n, (int)k, (int32_t*)sel.data_ptr(), st);
  });
  return failed(rc, "topk_select") ? nullptr : wrap(sel);
}

// (q bf16 [B, H, 128], keys e4m3 [B, N, 128], key_scales [B, N], weights [B, H]) -> float32 [B, N]
PyObject* indexer_scores_fp8(PyObject* const* a, Py_ssize_t nargs) {
  MSPR_NARGS(4)
  const Tensor *q = dense(a[0], 3, at::kBFloat16), *keys = dense(a[1], 3), *ks = dense(a[2], 2, at::kFloat),
               *w = dense(a[3], 2, at::kFloat);
  if (!q || !keys || !ks || !w || !here({q, keys, ks, w})) return none();
  if (keys->scalar_type() != at::kFloat8_e4m3fn && keys->scalar_type() != at::kByte) return none();
  const int64_t B = q->size(0), H = q->size(1), N = keys->size(1);
  if (B < 1 || H < 1 || H > 64 || N < 1 || q->size(2) != 128 || keys->size(0) != B || keys->size(2) != 128 ||
      ks->size(0) != B || ks->size(1) != N || w->size(0) != B || w->size(1) != H)
    return none();
  Tensor scores = empty({B, N}, at::kFloat, *q);
  const int rc = launch([&](void* st) {
    return mspr_indexer_scores_fp8(q->const_data_ptr(), keys->const_data_ptr(), (const float*)ks->const_data_ptr(),
                                   (const float*)w->const_data_ptr(), (int)B, (int)H, N, (float*)scores.data_ptr(), st);
  });
  return failed(rc, "indexer_scores_fp8") ? nullptr : wrap(scores);
}

// (q [1, H, 1, 128], pooled_qat f32 [1, N, 128], weights f32 [1, 1, H], scale) -> float32 [N]
PyObject* fused_qat_indexer_scores(PyObject* const* a, Py_ssize_t nargs) {
  MSPR_NARGS(4)
  const Tensor *q = dense(a[0], 4), *p = dense(a[1], 3, at::kFloat), *w = dense(a[2], 3, at::kFloat);
  float scale;
  if (!q || !p || !w || !real(a[3], &scale) || !here({q, p, w})) return none();
  const int code = type_code(q->scalar_type());
  const int64_t H = q->size(1), N = p->size(1);
  if (code == kNoType || q->size(0) != 1 || q->size(2) != 1 || q->size(3) != 128 || H < 1 || H > 64 || p->size(0) != 1 ||
      p->size(2) != 128 || N < 1 || w->size(0) != 1 || w->size(1) != 1 || w->size(2) != H)
    return none();
  Tensor scores = empty({N}, at::kFloat, *q);
  const int rc = launch([&](void* st) {
    return mspr_fused_qat_indexer_scores(q->const_data_ptr(), code, (int)H, (const float*)p->const_data_ptr(), N,
                                         (const float*)w->const_data_ptr(), scale, (float*)scores.data_ptr(), st);
  });
  return failed(rc, "fused_qat_indexer_scores") ? nullptr : wrap(scores);
}

// (q [B, H, T, 128], weights f32 [B, T, H], index_comp [B, P, 128], pos0, ratio) -> float32 [B, T, P]
PyObject* indexer_scores_tiled_live(PyObject* const* a, Py_ssize_t nargs) {
  MSPR_NARGS(5)
  const Tensor *q = dense(a[0], 4), *w = dense(a[1], 3, at::kFloat), *c = dense(a[2], 3);
  int pos0, ratio;
  if (!q || !w || !c || !whole32(a[3], &pos0) || !whole32(a[4], &ratio) || !here({q, w, c})) return none();
  const int code = type_code(q->scalar_type());
  const int64_t B = q->size(0), H = q->size(1), T = q->size(2), P = c->size(1);
  if ((code != MSPR_F32 && code != MSPR_F16) || c->scalar_type() != q->scalar_type() || q->size(3) != 128 ||
      c->size(0) != B || c->size(2) != 128 || w->size(0) != B || w->size(1) != T || w->size(2) != H || B < 1 || T < 1 ||
      P < 1 || H > 64)
    return none();
  Tensor scores = empty({B, T, P}, at::kFloat, *q);
  Tensor ws = scratch(mspr_indexer_scores_tiled_live_workspace_bytes((int)B, (int)H, (int)T, P), *q);
  const int rc = launch([&](void* st) {
    return mspr_indexer_scores_tiled_live_ws(q->const_data_ptr(), (const float*)w->const_data_ptr(), c->const_data_ptr(),
                                             code, (int)B, (int)H, (int)T, P, pos0, ratio, (float*)scores.data_ptr(),
                                             ws.data_ptr(), ws.nbytes(), st);
  });
  return failed(rc, "indexer_scores_tiled_live") ? nullptr : wrap(scores);
}

// ---------------------------------------------------------------------------------------------- DS4 attention

// (x [..., T, W], inv_freq f32 [32], offset, inverse, positions f32 or None, most rows) -> like x
PyObject* fused_partial_rope(PyObject* const* a, Py_ssize_t nargs) {
  MSPR_NARGS(6)
  const Tensor* inv = dense(a[1], 1, at::kFloat);
  int64_t offset, max_rows;
  if (!THPVariable_Check(a[0]) || !inv || inv->size(0) != 32 || !whole(a[2], &offset) || !PyBool_Check(a[3]) ||
      !whole(a[5], &max_rows))
    return none();
  const Tensor& x = THPVariable_Unpack(a[0]);
  if (!x.is_cuda() || x.dim() < 2 || !x.is_contiguous() || !here({&x, inv})) return none();
  const int code = type_code(x.scalar_type());
  const int64_t W = x.size(-1), T = x.size(-2);
  if (code == kNoType || W < 64 || W % 4 != 0 || x.numel() == 0) return none();
  const float* positions = nullptr;
  if (a[4] == Py_None) {
    if (offset < 0 || offset + T > ((int64_t)1 << 24)) return none();
  } else {
    if (!THPVariable_Check(a[4])) return none();
    const Tensor& p = THPVariable_Unpack(a[4]);
    if (!p.is_cuda() || !p.is_contiguous() || p.scalar_type() != at::kFloat || p.numel() != T || !here({&x, &p}))
      return none();
    positions = (const float*)p.const_data_ptr();
    offset = 0;
  }
  const int64_t rows = x.numel() / W;
  if (rows > max_rows || rows > 0x7FFFFFFF) return none();
  Tensor out = empty(x.sizes(), x.scalar_type(), x);
  const int inverse = a[3] == Py_True ? 1 : 0;
  const int rc = launch([&](void* st) {
    return mspr_fused_partial_rope(x.const_data_ptr(), code, rows / T, T, (int)W, (const float*)inv->const_data_ptr(),
                                   positions, offset, inverse, out.data_ptr(), st);
  });
  return failed(rc, "fused_partial_rope") ? nullptr : wrap(out);
}

// (q_idx [H, 128], pooled_qat f32 [N, 128], weights f32 [H], kv_row f16 [512], inv_freq f32 [32], params int32 [2+],
//  scale, topk, pool_rows_in_params) -> (sel int32 [topk], row f16 [512], scores f32 [N])
PyObject* fused_decode_prep(PyObject* const* a, Py_ssize_t nargs) {
  MSPR_NARGS(9)
  const Tensor *q = dense(a[0], 2), *p = dense(a[1], 2, at::kFloat), *w = dense(a[2], 1, at::kFloat),
               *kv = dense(a[3], 1, at::kHalf), *inv = dense(a[4], 1, at::kFloat), *prm = dense(a[5], 1, at::kInt);
  float scale;
  int64_t topk;
  if (!q || !p || !w || !kv || !inv || !prm || !real(a[6], &scale) || !whole(a[7], &topk) || !PyBool_Check(a[8]) ||
      !here({q, p, w, kv, inv, prm}))
    return none();
  const bool fixed = a[8] == Py_True;
  const int code = type_code(q->scalar_type());
  const int64_t H = q->size(0), N = p->size(0);
  if (code == kNoType || H < 1 || H > 64 || q->size(1) != 128 || p->size(1) != 128 || topk < 1 || topk >= N ||
      w->size(0) != H || kv->size(0) != 512 || inv->size(0) != 32 || prm->size(0) < (fixed ? 3 : 1))
    return none();
  Tensor sel = empty({topk}, at::kInt, *q), row = empty({512}, at::kHalf, *q), scores = empty({N}, at::kFloat, *q);
  const auto entry = fixed ? mspr_fused_decode_prep_fixed : mspr_fused_decode_prep;
  const int rc = launch([&](void* st) {
    return entry(q->const_data_ptr(), code, (int)H, (const float*)p->const_data_ptr(), N, (const float*)w->const_data_ptr(),
                 kv->const_data_ptr(), (const float*)inv->const_data_ptr(), (const int32_t*)prm->const_data_ptr(), scale,
                 (int)topk, (int32_t*)sel.data_ptr(), row.data_ptr(), (float*)scores.data_ptr(), st);
  });
  return failed(rc, "fused_decode_prep") ? nullptr : wrap_tuple(sel, row, scores);
}

// (q f16 [H, 512], window f16 [W, 512], row f16 [512], pooled f16 [N, 512], sel int32 [K], sinks f16 [H],
//  inv_freq f32 [32], params int32 [2+], scale, pool_rows_in_params, workspace) -> f16 [H, 512]
PyObject* fused_decode_sdpa(PyObject* const* a, Py_ssize_t nargs) {
  MSPR_NARGS(11)
  const Tensor *q = dense(a[0], 2, at::kHalf), *win = dense(a[1], 2, at::kHalf), *row = dense(a[2], 1, at::kHalf),
               *pool = dense(a[3], 2, at::kHalf), *sel = dense(a[4], 1, at::kInt), *sinks = dense(a[5], 1, at::kHalf),
               *inv = dense(a[6], 1, at::kFloat), *prm = dense(a[7], 1, at::kInt);
  float scale;
  if (!q || !win || !row || !pool || !sel || !sinks || !inv || !prm || !real(a[8], &scale) || !PyBool_Check(a[9]) ||
      !here({q, win, row, pool, sel, sinks, inv, prm}))
    return none();
  const bool fixed = a[9] == Py_True;
  const int64_t H = q->size(0), W = win->size(0), N = pool->size(0), K = sel->size(0);
  if (H < 1 || H > 4096 || q->size(1) != 512 || W < 1 || W > 0x3FFFFFFF || win->size(1) != 512 || row->size(0) != 512 ||
      pool->size(1) != 512 || K > 0x3FFFFFFF || sinks->size(0) != H || inv->size(0) != 32 || prm->size(0) < (fixed ? 3 : 2))
    return none();
  Tensor ws;
  if (!take_workspace(a[10], mspr_sparse_attention_workspace_bytes(1, (int)H, W + K), *q, &ws)) return none();
  Tensor out = empty({H, 512}, at::kHalf, *q);
  const auto entry = fixed ? mspr_fused_decode_sdpa_fixed : mspr_fused_decode_sdpa;
  const int rc = launch([&](void* st) {
    return entry(q->const_data_ptr(), (int)H, win->const_data_ptr(), (int)W, row->const_data_ptr(), pool->const_data_ptr(), N,
                 (const int32_t*)sel->const_data_ptr(), (int)K, sinks->const_data_ptr(), (const float*)inv->const_data_ptr(),
                 (const int32_t*)prm->const_data_ptr(), scale, out.data_ptr(), ws.data_ptr(), ws.nbytes(), st);
  });
  return failed(rc, "fused_decode_sdpa") ? nullptr : wrap(out);
}

// (q [B, H, D], kv [B, P, D], rows int32 [B, K], scale, v_dim, window_start or None, window_rows, sinks f32 [H] or None,
//  workspace, row_mul, row_add) -> [B, H, 512] like q
PyObject* sparse_mla_decode(PyObject* const* a, Py_ssize_t nargs) {
  MSPR_NARGS(11)
  const Tensor *q = dense(a[0], 3), *kv = dense(a[1], 3), *rows = dense(a[2], 2, at::kInt), *sinks = nullptr;
  float scale;
  int v_dim, win_rows, row_mul, row_add;
  int64_t win_start = 0;
  if (!q || !kv || !rows || !real(a[3], &scale) || !whole32(a[4], &v_dim) || !whole32(a[6], &win_rows) ||
      !whole32(a[9], &row_mul) || !whole32(a[10], &row_add) || !here({q, kv, rows}))
    return none();
  if (a[5] != Py_None && !whole(a[5], &win_start)) return none();
  const int64_t B = q->size(0), H = q->size(1), D = q->size(2), P = kv->size(1), K = rows->size(1);
  if (a[7] != Py_None) {
    sinks = dense(a[7], 1, at::kFloat);
    if (!sinks || sinks->size(0) != H || !here({q, sinks})) return none();
  }
  if ((q->scalar_type() != at::kHalf && q->scalar_type() != at::kBFloat16) || kv->scalar_type() != q->scalar_type() ||
      B < 1 || B > 65535 || H < 1 || H > 128 || (D != 512 && D != 576) || v_dim != 512 || kv->size(0) != B ||
      kv->size(2) != D || rows->size(0) != B || K > 0x3FFFFFFF || win_rows < 0 ||
      (win_rows > 0 && (win_start < 0 || win_start + win_rows > P)))
    return none();
  Tensor ws;
  if (!take_workspace(a[8], mspr_sparse_attention_workspace_bytes((int)B, (int)H, K + win_rows), *q, &ws)) return none();
  Tensor out = empty({B, H, 512}, q->scalar_type(), *q);
  const int rc = launch([&](void* st) {
    return mspr_sparse_mla_decode(q->const_data_ptr(), kv->const_data_ptr(), (const int32_t*)rows->const_data_ptr(),
                                  (const float*)at_or_null(sinks), type_code(q->scalar_type()), (int)B, (int)H, (int)D, 512,
                                  P, (int)K, row_mul, row_add, win_start, win_rows, scale, out.data_ptr(), ws.data_ptr(),
                                  ws.nbytes(), st);
  });
  return failed(rc, "sparse_mla_decode") ? nullptr : wrap(out);
}

// (q [B, H, T, 512] f16 or f32, raw_kv f16 [B, 1, R, 512], comp_kv f16 [B, P, 512], topk int32 [B, T, K], sinks f32 [H],
//  pos0, window, ratio, raw_start) -> float32 like q; the operands have been validated
PyObject* prefill_live(PyObject* const* a, Py_ssize_t nargs) {
  MSPR_NARGS(9)
  const Tensor *q = dense(a[0], 4), *raw = dense(a[1], 4, at::kHalf), *comp = dense(a[2], 3, at::kHalf),
               *topk = dense(a[3], 3, at::kInt), *sinks = dense(a[4], 1, at::kFloat);
  int pos0, window, ratio, raw_start;
  if (!q || !raw || !comp || !topk || !sinks || !whole32(a[5], &pos0) || !whole32(a[6], &window) ||
      !whole32(a[7], &ratio) || !whole32(a[8], &raw_start) || !here({q, raw, comp, topk, sinks}))
    return none();
  const int code = type_code(q->scalar_type());
  const int64_t B = q->size(0), H = q->size(1), T = q->size(2), R = raw->size(2), P = comp->size(1), K = topk->size(2);
  if ((code != MSPR_F16 && code != MSPR_F32) || q->size(3) != 512 || raw->size(0) != B || raw->size(1) != 1 ||
      raw->size(3) != 512 || comp->size(0) != B || comp->size(2) != 512 || topk->size(0) != B || topk->size(1) != T ||
      sinks->size(0) != H || R > 0x7FFFFFFF || K > 0x7FFFFFFF)
    return none();
  const int max_win = window != 0 && window < R ? window : (int)R;
  Tensor ws = scratch(mspr_indexed_mixed_attention_prefill_workspace_bytes(code, (int)B, (int)H, (int)T, max_win, (int)K), *q);
  Tensor out = empty(q->sizes(), at::kFloat, *q);
  const int rc = launch([&](void* st) {
    return mspr_indexed_mixed_attention_prefill(
        q->const_data_ptr(), code, (int)B, (int)H, (int)T, H * T * 512, T * 512, 512, raw->const_data_ptr(), (int)R,
        comp->const_data_ptr(), P, K ? (const int32_t*)topk->const_data_ptr() : nullptr, (int)K,
        (const float*)sinks->const_data_ptr(), pos0, window, ratio, raw_start, (float*)out.data_ptr(), ws.data_ptr(),
        ws.nbytes(), st);
  });
  return failed(rc, "indexed_mixed_attention_prefill") ? nullptr : wrap(out);
}

// ---------------------------------------------------------------------------------------------- Qwen, 8-bit cache

// (x [..., D]) -> (wq uint32 [..., D/4], scales [..., D/64], biases [..., D/64])
PyObject* quantize(PyObject* const* a, Py_ssize_t nargs) {
  MSPR_NARGS(1)
  if (!THPVariable_Check(a[0])) return none();
  const Tensor& x = THPVariable_Unpack(a[0]);
  if (!here(x) || x.dim() < 1 || x.numel() == 0 || !x.is_contiguous() || x.size(-1) % 64 != 0) return none();
  const int code = type_code(x.scalar_type());
  if (code == kNoType) return none();
  at::DimVector shape(x.sizes());
  shape.back() = x.size(-1) / 4;
  Tensor wq = empty(shape, at::kUInt32, x);
  shape.back() = x.size(-1) / 64;
  Tensor scales = empty(shape, x.scalar_type(), x), biases = empty(shape, x.scalar_type(), x);
  const int rc = launch([&](void* st) {
    return mspr_affine_q8_quantize(x.const_data_ptr(), code, x.numel() / 64, wq.data_ptr(), scales.data_ptr(),
                                   biases.data_ptr(), 64, 8, st);
  });
  return failed(rc, "quantize") ? nullptr : wrap_tuple(wq, scales, biases);
}

// (wq uint32 [..., D/4], scales, biases [..., D/64]) -> [..., D] like scales
PyObject* dequantize(PyObject* const* a, Py_ssize_t nargs) {
  MSPR_NARGS(3)
  for (int i = 0; i < 3; i++)
    if (!THPVariable_Check(a[i])) return none();
  const Tensor &w = THPVariable_Unpack(a[0]), &s = THPVariable_Unpack(a[1]), &b = THPVariable_Unpack(a[2]);
  if (!w.is_cuda() || !s.is_cuda() || !b.is_cuda() || !w.is_contiguous() || !s.is_contiguous() || !b.is_contiguous())
    return none();
  const int code = type_code(s.scalar_type());
  if (code == kNoType || b.scalar_type() != s.scalar_type() || w.numel() == 0 || w.dim() < 1 || w.dim() != s.dim() ||
      s.sizes() != b.sizes() || (w.scalar_type() != at::kUInt32 && w.scalar_type() != at::kInt) || !here({&w, &s, &b}))
    return none();
  at::DimVector shape(w.sizes());
  for (int64_t d = 0; d + 1 < w.dim(); d++)
    if (w.size(d) != s.size(d)) return none();
  if (w.size(-1) != 16 * s.size(-1)) return none();
  shape.back() = w.size(-1) * 4;
  Tensor out = empty(shape, s.scalar_type(), s);
  const int rc = launch([&](void* st) {
    return mspr_affine_q8_dequantize(w.const_data_ptr(), s.const_data_ptr(), b.const_data_ptr(), code, s.numel(),
                                     out.data_ptr(), 64, 8, st);
  });
  return failed(rc, "dequantize") ? nullptr : wrap(out);
}

// Row capacity of [B, H, N, W] tensors that are the leading rows of every head of dense [B, H, capacity, W] buffers,
// the same for all of them (what a cache that grows in blocks hands out); -1 if they are not.
int64_t common_row_capacity(std::initializer_list<const Tensor*> ts) {
  int64_t common = -2;
  for (const Tensor* t : ts) {
    const int64_t B = t->size(0), H = t->size(1), N = t->size(2), W = t->size(3);
    if (W < 1 || t->stride(3) != 1 || t->stride(2) != W) return -1;
    int64_t cap = N;
    if (B * H > 1) {
      cap = (H > 1 ? t->stride(1) : t->stride(0)) / W;
      if (cap < N || (H > 1 && t->stride(1) != cap * W) || (B > 1 && t->stride(0) != H * cap * W)) return -1;
    }
    if (common != -2 && cap != common) return -1;
    common = cap;
  }
  return common;
}

// A 4-D tensor on a HIP device whose layout the capacity rule above judges.
const Tensor* cache_part(PyObject* o) {
  if (!THPVariable_Check(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  return t.is_cuda() && t.dim() == 4 ? &t : nullptr;
}

// Codes [B, Hkv, N, 64] of 32-bit words with scales and biases [B, Hkv, N, 4], keys and values alike.
bool affine_cache(PyObject* const* a, const Tensor* (&t)[6], int64_t B, int64_t* Hkv, int64_t* N, int* sb_code, int64_t* cap) {
  for (int i = 0; i < 6; i++)
    if (!(t[i] = cache_part(a[i]))) return false;
  *Hkv = t[0]->size(1);
  *N = t[0]->size(2);
  *sb_code = type_code(t[1]->scalar_type());
  if (*sb_code == kNoType || *Hkv < 1 || *Hkv > 4096) return false;
  for (int i = 0; i < 6; i++) {
    const bool codes = i % 3 == 0;
    if (t[i]->size(0) != B || t[i]->size(1) != *Hkv || t[i]->size(2) != *N || t[i]->size(3) != (codes ? 64 : 4)) return false;
    if (codes ? (t[i]->scalar_type() != at::kUInt32 && t[i]->scalar_type() != at::kInt)
              : t[i]->scalar_type() != t[1]->scalar_type())
      return false;
  }
  if (!here({t[0], t[1], t[2], t[3], t[4], t[5]})) return false;
  *cap = common_row_capacity({t[0], t[1], t[2], t[3], t[4], t[5]});
  return *cap >= *N;
}

// The three tensors of a cache side, capacity buffers [B, H, cap, *].
bool cache_side(PyObject* o, const Tensor* (&t)[3]) {
  if (!PyTuple_CheckExact(o) || PyTuple_GET_SIZE(o) != 3) return false;
  for (int i = 0; i < 3; i++)
    if (!(t[i] = cache_part(PyTuple_GET_ITEM(o, i)))) return false;
  return true;
}

// both sides as views of the first n rows of every head
PyObject* wrap_leading_rows(const Tensor* const (&t)[2][3], int64_t n) {
  PyObject* sides[2];
  for (int s = 0; s < 2; s++) {
    sides[s] = wrap_tuple(t[s][0]->slice(2, 0, n), t[s][1]->slice(2, 0, n), t[s][2]->slice(2, 0, n));
    if (!sides[s]) return nullptr;
  }
  PyObject* r = PyTuple_Pack(2, sides[0], sides[1]);
  Py_DECREF(sides[0]);
  Py_DECREF(sides[1]);
  return r;
}

// (keys [B, H, L, D], values, key side, value side, offset): quantises the rows into the buffers of both sides behind the
// first `offset` rows of every head -> ((key side, value side) up to the new length, the new length)
PyObject* q8_append(PyObject* const* a, Py_ssize_t nargs) {
  MSPR_NARGS(5)
  const Tensor *k = dense(a[0], 4), *v = dense(a[1], 4), *side[2][3];
  int64_t offset;
  if (!k || !v || !cache_side(a[2], side[0]) || !cache_side(a[3], side[1]) || !whole(a[4], &offset)) return none();
  const Tensor *const(&ks)[3] = side[0], *const(&vs)[3] = side[1];
  const int code = type_code(k->scalar_type());
  const int64_t B = k->size(0), H = k->size(1), L = k->size(2), D = k->size(3), cap = ks[0]->size(2);
  if (code == kNoType || v->scalar_type() != k->scalar_type() || k->sizes() != v->sizes() || k->numel() == 0 || D % 64 != 0 ||
      D > 4096 || B * H > 65535 || offset < 0 || offset + L > cap || !here({k, v, ks[0], ks[1], ks[2], vs[0], vs[1], vs[2]}))
    return none();
  for (const auto& half : side)
    for (int i = 0; i < 3; i++) {
      const Tensor& t = *half[i];
      const bool codes = i == 0;
      if (!t.is_contiguous() || t.size(0) != B || t.size(1) != H || t.size(2) != cap || t.size(3) != (codes ? D / 4 : D / 64) ||
          t.scalar_type() != (codes ? at::kUInt32 : k->scalar_type()))
        return none();
    }
  const int rc = launch([&](void* st) {
    return mspr_affine_q8_append(k->const_data_ptr(), v->const_data_ptr(), code, (int)(B * H), L, (int)D, ks[0]->data_ptr(),
                                 ks[1]->data_ptr(), ks[2]->data_ptr(), vs[0]->data_ptr(), vs[1]->data_ptr(),
                                 vs[2]->data_ptr(), cap, offset, st);
  });
  if (failed(rc, "q8_append")) return nullptr;
  PyObject* views = wrap_leading_rows(side, offset + L);
  PyObject* length = views ? PyLong_FromLongLong(offset + L) : nullptr;
  PyObject* r = length ? PyTuple_Pack(2, views, length) : nullptr;
  Py_XDECREF(views);
  Py_XDECREF(length);
  return r;
}

// (key side, value side, n) -> both sides as views of the first n rows of every head
PyObject* leading_rows(PyObject* const* a, Py_ssize_t nargs) {
  MSPR_NARGS(3)
  const Tensor* t[2][3];
  int64_t n;
  if (!cache_side(a[0], t[0]) || !cache_side(a[1], t[1]) || !whole(a[2], &n)) return none();
  for (const auto& side : t)
    for (const Tensor* p : side)
      if (n < 0 || n > p->size(2)) return none();
  return wrap_leading_rows(t, n);
}

// (queries f32 [B, Hq, 1, 256], six cache parts, scale, workspace) -> f32 like queries
PyObject* sdpa_decode_q8(PyObject* const* a, Py_ssize_t nargs) {
  MSPR_NARGS(9)
  const Tensor *q = dense(a[0], 4, at::kFloat), *t[6];
  float scale;
  if (!q || q->size(2) != 1 || q->size(3) != 256 || !real(a[7], &scale)) return none();
  const int64_t B = q->size(0), Hq = q->size(1);
  int64_t Hkv, N, cap;
  int sb;
  if (!affine_cache(a + 1, t, B, &Hkv, &N, &sb, &cap) || N < 1 || B < 1 || B > 65535 || Hq < 1 || Hq % Hkv != 0 ||
      Hq / Hkv > 16 || !here({q, t[0]}))
    return none();
  Tensor ws;
  if (!take_workspace(a[8], mspr_sdpa_decode_q8_workspace_bytes((int)B, (int)Hkv, N), *q, &ws)) return none();
  Tensor out = empty(q->sizes(), at::kFloat, *q);
  const int rc = launch([&](void* st) {
    return mspr_sdpa_decode_q8(q->const_data_ptr(), MSPR_F32, t[0]->const_data_ptr(), t[1]->const_data_ptr(),
                               t[2]->const_data_ptr(), t[3]->const_data_ptr(), t[4]->const_data_ptr(),
                               t[5]->const_data_ptr(), sb, (int)B, (int)Hq, (int)Hkv, 256, N, cap, scale, 64, 8,
                               out.data_ptr(), ws.data_ptr(), ws.nbytes(), st);
  });
  return failed(rc, "sdpa_decode_q8") ? nullptr : wrap(out);
}

// (queries [B, Hq, 256], k_codes int8 [B, Hkv, N, 256], k_scales f16 [B, Hkv, N, 8], v_codes, v_scales, scale, workspace)
PyObject* sdpa_decode_q8_0(PyObject* const* a, Py_ssize_t nargs) {
  MSPR_NARGS(7)
  const Tensor *q = dense(a[0], 3), *kc = cache_part(a[1]), *ks = cache_part(a[2]), *vc = cache_part(a[3]),
               *vs = cache_part(a[4]);
  float scale;
  if (!q || !kc || !ks || !vc || !vs || !real(a[5], &scale) || !here({q, kc, ks, vc, vs})) return none();
  const int code = type_code(q->scalar_type());
  const int64_t B = q->size(0), Hq = q->size(1), Hkv = kc->size(1), N = kc->size(2);
  if (code == kNoType || q->size(2) != 256 || B < 1 || B > 65535 || Hkv < 1 || Hq < 1 || Hq % Hkv != 0 || Hq / Hkv > 16 ||
      N < 1 || kc->scalar_type() != at::kChar || vc->scalar_type() != at::kChar || ks->scalar_type() != at::kHalf ||
      vs->scalar_type() != at::kHalf || kc->size(0) != B || kc->size(3) != 256 || kc->sizes() != vc->sizes() ||
      ks->size(0) != B || ks->size(1) != Hkv || ks->size(2) != N || ks->size(3) != 8 || ks->sizes() != vs->sizes())
    return none();
  const int64_t cap = common_row_capacity({kc, ks, vc, vs});
  if (cap < N) return none();
  Tensor ws;
  if (!take_workspace(a[6], mspr_sdpa_decode_q8_workspace_bytes((int)B, (int)Hkv, N), *q, &ws)) return none();
  Tensor out = empty(q->sizes(), q->scalar_type(), *q);
  const int rc = launch([&](void* st) {
    return mspr_sdpa_decode_q8_0(q->const_data_ptr(), code, kc->const_data_ptr(), ks->const_data_ptr(),
                                 vc->const_data_ptr(), vs->const_data_ptr(), (int)B, (int)Hq, (int)Hkv, 256, N, cap, scale,
                                 out.data_ptr(), ws.data_ptr(), ws.nbytes(), st);
  });
  return failed(rc, "sdpa_decode_q8_0") ? nullptr : wrap(out);
}

// (queries f32 [B, Hq, L, 256], six prefix parts, self_k, self_v [B, Hkv, L, 256], scale, workspace) -> f32 like queries
PyObject* sdpa_fa_prefill_q8(PyObject* const* a, Py_ssize_t nargs) {
  MSPR_NARGS(11)
  const Tensor *q = dense(a[0], 4, at::kFloat), *sk = dense(a[7], 4), *sv = dense(a[8], 4), *t[6];
  float scale;
  if (!q || !sk || !sv || q->size(3) != 256 || !real(a[9], &scale)) return none();
  const int64_t B = q->size(0), Hq = q->size(1), L = q->size(2);
  int64_t Hkv, P, cap;
  int sb;
  const int self_code = type_code(sk->scalar_type());
  if (!affine_cache(a + 1, t, B, &Hkv, &P, &sb, &cap) || self_code == kNoType || sv->scalar_type() != sk->scalar_type() ||
      sk->sizes() != sv->sizes() || sk->size(0) != B || sk->size(1) != Hkv || sk->size(2) != L || sk->size(3) != 256 ||
      B < 1 || L < 1 || L > 0x7FFFFFFF || Hq < 1 || Hq > 4096 || !here({q, t[0], sk, sv}))
    return none();
  const int64_t rep = Hq / Hkv;
  if (Hq % Hkv != 0 || (rep != 1 && rep != 2 && rep != 4 && rep != 8)) return none();
  Tensor ws;
  if (!take_workspace(a[10], mspr_sdpa_fa_prefill_q8_workspace_bytes((int)B, (int)Hq, (int)Hkv, (int)L, P), *q, &ws))
    return none();
  Tensor out = empty(q->sizes(), at::kFloat, *q);
  const int rc = launch([&](void* st) {
    return mspr_sdpa_fa_prefill_q8(q->const_data_ptr(), t[0]->const_data_ptr(), t[1]->const_data_ptr(),
                                   t[2]->const_data_ptr(), t[3]->const_data_ptr(), t[4]->const_data_ptr(),
                                   t[5]->const_data_ptr(), sb, sk->const_data_ptr(), sv->const_data_ptr(), self_code, (int)B,
                                   (int)Hq, (int)Hkv, 256, (int)L, P, cap, scale, 64, 8, out.data_ptr(), ws.data_ptr(),
                                   ws.nbytes(), st);
  });
  return failed(rc, "sdpa_fa_prefill_q8") ? nullptr : wrap(out);
}

PyMethodDef kMethods[] = {
#define MSPR_METHOD(name) {#name, (PyCFunction)(void (*)(void))guarded<name>, METH_FASTCALL, nullptr}
    {"indexer_qat_rows", (PyCFunction)(void (*)(void))guarded<qat_rows<false>>, METH_FASTCALL, nullptr},
    {"indexer_q_qat_live", (PyCFunction)(void (*)(void))guarded<qat_rows<true>>, METH_FASTCALL, nullptr},
    MSPR_METHOD(topk_select),
    MSPR_METHOD(indexer_scores_fp8),
    MSPR_METHOD(fused_qat_indexer_scores),
    MSPR_METHOD(indexer_scores_tiled_live),
    MSPR_METHOD(fused_partial_rope),
    MSPR_METHOD(fused_decode_prep),
    MSPR_METHOD(fused_decode_sdpa),
    MSPR_METHOD(sparse_mla_decode),
    MSPR_METHOD(prefill_live),
    MSPR_METHOD(quantize),
    MSPR_METHOD(dequantize),
    MSPR_METHOD(q8_append),
    MSPR_METHOD(leading_rows),
    MSPR_METHOD(sdpa_decode_q8),
    MSPR_METHOD(sdpa_decode_q8_0),
    MSPR_METHOD(sdpa_fa_prefill_q8),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_dispatch", "Native call path of the operators.", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__dispatch(void) {
  PyObject* m = PyModule_Create(&kModule);
  if (m && PyModule_AddStringConstant(m, "torch_version", MSPR_TORCH_VERSION) != 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
