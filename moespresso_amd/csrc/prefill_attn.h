// Launch interface of the indexed prefill attention kernel (prefill_attn.hip).
#pragma once
#include "common.h"

// What the kernel reads behind its plain arguments. (The last four words come in one load and are all used late: the register
// of a word that is not is given away, and its next owner waits for the load.)
struct IndexedPrefillRest {
  const void* q;  // element (b, t, head, d) at b*q_batch_stride + t*q_token_stride + head*q_head_stride + d
  int64_t q_batch_stride, q_head_stride, q_token_stride;
  const void* pool;  // float16 [batch][n_pool][512]
  const float* sinks;  // [n_heads] or null
  float* out;  // strides as q
  float* parts;  // filled in by the launch: partials of the units that are cut into key ranges
  int n_heads;
  uint32_t ratio;
  int n_pool;
  float scale_log2;
};

struct IndexedPrefillArgs : IndexedPrefillRest {
  int q_dtype;    // MSPR_F16 or MSPR_F32 (rounded to float16 on load)
  int batch, n_tokens;
  const void* win;  // float16 ring [batch][raw_cap][512]
  int raw_cap, raw_start;
  int max_win;      // most ring rows any token visits
  const int32_t* idx;  // [batch][n_tokens][n_idx]
  int n_idx;
  uint32_t pos0, window;
  // filled in by the launch: units (token and block of 64 heads) that are cut into key ranges
  int split_units, ranges;
};

// Whether the kernel takes the call: the ids of a token are staged in LDS next to the row tiles.
bool mspr_indexed_prefill_fits(int batch, int n_heads, int n_tokens, int n_idx);
// Room for the partials of a part-filled last round; without it every token is one workgroup's.
size_t mspr_indexed_prefill_workspace_bytes(int batch, int n_heads, int n_tokens, int window_rows, int n_idx);
int mspr_launch_indexed_prefill(const IndexedPrefillArgs& a, void* workspace, size_t workspace_bytes, hipStream_t st);
