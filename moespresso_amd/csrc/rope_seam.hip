// Partial rotary embedding of the last 64 channels of rows laid out [..., seq, width]; the leading
// channels copy through. One pass replaces the composed split / angle table / cos / sin / four
// multiplies / stack / concat sequence, with that sequence's rounding: the angle is one float32
// multiply position * inv_freq[p]; cos and sin are taken at float32 and cast to the element type (the
// inverse form negates the float32 sine first); every product and every sum of the rotation is
// rounded to the element type on its own (float32 rows: float32 operations, never contracted).
//
// A workgroup owns one sequence position (the wide form below: a few) and a slab of the outer rows (batch x heads): the
// cosine / sine pairs of the position are worked out once and shared through LDS, so the transcendental work does not
// grow with the head count; the rows then stream through. Both forms are bound by memory.
#include "common.h"

#pragma clang fp contract(off)

namespace {

constexpr int kRopeDim = 64;
constexpr int kRopeFreqs = kRopeDim / 2;
constexpr int kThreads = 256;

template <int DT>
__device__ __forceinline__ float round_to(float v) {
  if constexpr (DT == MSPR_F32) return v;
  else if constexpr (DT == MSPR_F16) return f16_bits_to_f32(f32_to_f16_bits(v));
  else return bf16_bits_to_f32(f32_to_bf16_bits(v));
}

template <int DT>
__device__ __forceinline__ f32x4_t load_quad(const void* p, int64_t quad) {
  if constexpr (DT == MSPR_F32) {
    return reinterpret_cast<const f32x4_t*>(p)[quad];
  } else {
    const u32x2_t w = reinterpret_cast<const u32x2_t*>(p)[quad];
    if constexpr (DT == MSPR_F16)
      return f32x4_t{f16_bits_to_f32((uint16_t)(w.x & 0xFFFFu)), f16_bits_to_f32((uint16_t)(w.x >> 16)),
                     f16_bits_to_f32((uint16_t)(w.y & 0xFFFFu)), f16_bits_to_f32((uint16_t)(w.y >> 16))};
    else
      return f32x4_t{bf16_bits_to_f32((uint16_t)(w.x & 0xFFFFu)), bf16_bits_to_f32((uint16_t)(w.x >> 16)),
                     bf16_bits_to_f32((uint16_t)(w.y & 0xFFFFu)), bf16_bits_to_f32((uint16_t)(w.y >> 16))};
  }
}

template <int DT>
__device__ __forceinline__ void store_quad(void* p, int64_t quad, f32x4_t v) {
  if constexpr (DT == MSPR_F32) {
    reinterpret_cast<f32x4_t*>(p)[quad] = v;
  } else if constexpr (DT == MSPR_F16) {
    reinterpret_cast<u32x2_t*>(p)[quad] =
        u32x2_t{(uint32_t)f32_to_f16_bits(v.x) | ((uint32_t)f32_to_f16_bits(v.y) << 16),
                (uint32_t)f32_to_f16_bits(v.z) | ((uint32_t)f32_to_f16_bits(v.w) << 16)};
  } else {
    reinterpret_cast<u32x2_t*>(p)[quad] =
        u32x2_t{(uint32_t)f32_to_bf16_bits(v.x) | ((uint32_t)f32_to_bf16_bits(v.y) << 16),
                (uint32_t)f32_to_bf16_bits(v.z) | ((uint32_t)f32_to_bf16_bits(v.w) << 16)};
  }
}

// grid: (seq_len, slabs); a slab is `rows_per_wg` outer rows
template <int DT>
__global__ __launch_bounds__(kThreads) void partial_rope_kernel(const void* __restrict__ x, int64_t n_outer,
                                                               int64_t seq_len, int width,
                                                               const float* __restrict__ inv_freq,
                                                               const float* __restrict__ positions, int64_t offset,
                                                               int inverse, int rows_per_wg, void* __restrict__ out) {
  __shared__ float cs[kRopeFreqs], sn[kRopeFreqs];
  const int tid = threadIdx.x;
  const int64_t l = blockIdx.x;
  if (tid < kRopeFreqs) {
    const float pos = positions ? positions[l] : (float)(offset + l);
    const float theta = pos * inv_freq[tid];
    // float32 cosine and sine of the float32 angle, correctly rounded
    const float c = (float)cos((double)theta);
    float s = (float)sin((double)theta);
    if (inverse) s = -s;
    cs[tid] = round_to<DT>(c);
    sn[tid] = round_to<DT>(s);
  }
  __syncthreads();

  const int quads = width / 4;
  const int tail_quad = (width - kRopeDim) / 4;
  const int64_t o0 = (int64_t)blockIdx.y * rows_per_wg;
  int64_t o1 = o0 + rows_per_wg;
  if (o1 > n_outer) o1 = n_outer;
  const int64_t items = (o1 - o0) * quads;
  for (int64_t it = tid; it < items; it += kThreads) {
    const int64_t o = o0 + it / quads;
    const int qd = (int)(it % quads);
    const int64_t quad = (o * seq_len + l) * quads + qd;
    f32x4_t v = load_quad<DT>(x, quad);
    if (qd >= tail_quad) {
      const int p = 2 * (qd - tail_quad);  // first of the two pairs of this quad
      f32x4_t r;
      {
        const float c = cs[p], s = sn[p];
        const float m0 = round_to<DT>(v.x * c), m1 = round_to<DT>(v.y * s);
        const float m2 = round_to<DT>(v.x * s), m3 = round_to<DT>(v.y * c);
        r.x = round_to<DT>(m0 - m1);
        r.y = round_to<DT>(m2 + m3);
      }
      {
        const float c = cs[p + 1], s = sn[p + 1];
        const float m0 = round_to<DT>(v.z * c), m1 = round_to<DT>(v.w * s);
        const float m2 = round_to<DT>(v.z * s), m3 = round_to<DT>(v.w * c);
        r.z = round_to<DT>(m0 - m1);
        r.w = round_to<DT>(m2 + m3);
      }
      v = r;
    }
    store_quad<DT>(out, quad, v);
  }
}

// Wide form, for rows of whole 16-byte chunks that divide the workgroup (64 to 1024 channels of 16 bits, 64 to 512 of
// 32): the workgroup covers kThreads chunks = kThreads / chunks-per-row consecutive positions of one outer row at a time,
// 4 KB of contiguous memory, and walks its slab of outer rows at the same positions. A thread keeps its place in the row
// and its position, so its cosines and sines stay in registers and no index arithmetic is left in the loop.
// STREAM: the rows are read past the caches. STORE: how they are written (see store_window). Bound by memory: 3844 tokens
// of 64 x 512 rows, fresh ones each call, 504 MB of float16 in and out 112 us cached, 85 read and written as streams, 77.5
// read as a stream and written through; 1008 MB of float32 174 (read as a stream) and 169; 126 MB of float32 39.5 and 37.4;
// 517 tokens of 64 x 512 in float32 22.6 and 21.4, in float16 12.0 and 12.2. (Written through and as a stream 1008 MB take
// 162, but what reads them next more than that; 126 MB 41.7.)
template <int DT, bool STREAM, int STORE>
__global__ __launch_bounds__(kThreads) void partial_rope_wide_kernel(const void* __restrict__ x, int n_outer, int seq_len,
                                                                    int chunks_log2, const float* __restrict__ inv_freq,
                                                                    const float* __restrict__ positions, int64_t offset,
                                                                    int inverse, int rows_per_wg, void* __restrict__ out) {
  constexpr int kPairs = DT == MSPR_F32 ? 2 : 4;  // of a 16-byte chunk
  constexpr int kMaxPos = kThreads * kPairs * 2 / kRopeDim;
  __shared__ float cs[kMaxPos * kRopeFreqs], sn[kMaxPos * kRopeFreqs];
  const int tid = threadIdx.x;
  const int n_pos = kThreads >> chunks_log2;
  const int l0 = blockIdx.x * n_pos;
  for (int i = tid; i < n_pos * kRopeFreqs; i += kThreads) {
    const int l = l0 + i / kRopeFreqs;
    const float pos = positions ? positions[l < seq_len ? l : seq_len - 1] : (float)(offset + l);
    const float theta = pos * inv_freq[i % kRopeFreqs];
    // float32 cosine and sine of the float32 angle, correctly rounded
    const float c = (float)cos((double)theta);
    float s = (float)sin((double)theta);
    if (inverse) s = -s;
    cs[i] = round_to<DT>(c);
    sn[i] = round_to<DT>(s);
  }
  __syncthreads();
  const int chunk = tid & ((1 << chunks_log2) - 1), lp = tid >> chunks_log2;
  if (l0 + lp >= seq_len) return;
  const int tail_chunk = (1 << chunks_log2) - kRopeDim / (2 * kPairs);
  const bool tail = chunk >= tail_chunk;
  float c[kPairs], s[kPairs];
#pragma unroll
  for (int p = 0; p < kPairs; p++) {
    const int f = lp * kRopeFreqs + (tail ? (chunk - tail_chunk) * kPairs + p : 0);
    c[p] = cs[f];
    s[p] = sn[f];
  }
  const int64_t row_step = (int64_t)seq_len << chunks_log2;  // chunks between outer rows at one position
  int o = blockIdx.y * rows_per_wg;
  int n = n_outer - o;
  if (n > rows_per_wg) n = rows_per_wg;
  const u32x4_t* src = reinterpret_cast<const u32x4_t*>(x) + o * row_step + ((int64_t)(l0 + lp) << chunks_log2) + chunk;
  // (chunk tid of the workgroup's 4 KB in every outer row)
  unsigned char* dst = reinterpret_cast<unsigned char*>(out) + 16 * (o * row_step + ((int64_t)l0 << chunks_log2));
  auto pair = [&](float x0, float x1, int p, float* y0, float* y1) {
    const float m0 = round_to<DT>(x0 * c[p]), m1 = round_to<DT>(x1 * s[p]);
    const float m2 = round_to<DT>(x0 * s[p]), m3 = round_to<DT>(x1 * c[p]);
    *y0 = round_to<DT>(m0 - m1);
    *y1 = round_to<DT>(m2 + m3);
  };
  auto rotate = [&](u32x4_t v) -> u32x4_t {
#pragma unroll
    for (int p = 0; p < kPairs; p++) {
      float y0, y1;
      if constexpr (DT == MSPR_F32) {
        pair(__uint_as_float(v[2 * p]), __uint_as_float(v[2 * p + 1]), p, &y0, &y1);
        v[2 * p] = __float_as_uint(y0);
        v[2 * p + 1] = __float_as_uint(y1);
      } else if constexpr (DT == MSPR_F16) {
        pair(f16_bits_to_f32((uint16_t)(v[p] & 0xFFFFu)), f16_bits_to_f32((uint16_t)(v[p] >> 16)), p, &y0, &y1);
        v[p] = (uint32_t)f32_to_f16_bits(y0) | ((uint32_t)f32_to_f16_bits(y1) << 16);
      } else {
        pair(bf16_bits_to_f32((uint16_t)(v[p] & 0xFFFFu)), bf16_bits_to_f32((uint16_t)(v[p] >> 16)), p, &y0, &y1);
        v[p] = (uint32_t)f32_to_bf16_bits(y0) | ((uint32_t)f32_to_bf16_bits(y1) << 16);
      }
    }
    return v;
  };
  auto get = [](const u32x4_t* p) -> u32x4_t {
    if constexpr (STREAM) return __builtin_nontemporal_load(p);
    else return *p;
  };
  auto put = [&](u32x4_t v, unsigned char* row) { window_store<STORE>(store_window(row, 16 * kThreads), 16 * tid, v); };
  constexpr int kAtOnce = 4;  // rows in flight per thread
  for (; n >= kAtOnce; n -= kAtOnce) {
    u32x4_t v[kAtOnce];
#pragma unroll
    for (int j = 0; j < kAtOnce; j++) v[j] = get(src + j * row_step);
#pragma unroll
    for (int j = 0; j < kAtOnce; j++) {
      if (tail) v[j] = rotate(v[j]);
      put(v[j], dst + 16 * j * row_step);
    }
    src += kAtOnce * row_step;
    dst += 16 * kAtOnce * row_step;
  }
  for (; n > 0; n--) {
    u32x4_t v = get(src);
    if (tail) v = rotate(v);
    put(v, dst);
    src += row_step;
    dst += 16 * row_step;
  }
}

}  // namespace

extern "C" int mspr_fused_partial_rope(const void* x, int dtype, int64_t n_outer, int64_t seq_len, int width,
                                       const float* inv_freq, const float* positions, int64_t offset, int inverse,
                                       void* out, void* stream) {
  MSPR_REQUIRE(x && inv_freq && out, "fused_partial_rope: null pointer");
  MSPR_REQUIRE(dtype == MSPR_F32 || dtype == MSPR_F16 || dtype == MSPR_BF16,
               "fused_partial_rope: rows must be float32, float16, or bfloat16");
  MSPR_REQUIRE(n_outer >= 1 && seq_len >= 1, "fused_partial_rope: at least one row");
  MSPR_REQUIRE(seq_len <= 0x7FFFFFFF && n_outer * seq_len <= 0x7FFFFFFF, "fused_partial_rope: too many rows");
  MSPR_REQUIRE(width >= kRopeDim && width % 4 == 0, "fused_partial_rope: width must be a multiple of 4 and at least 64");
  MSPR_REQUIRE(positions || (offset >= 0 && offset + seq_len <= ((int64_t)1 << 24)),
               "fused_partial_rope: positions must stay exact in float32");
  MSPR_REQUIRE(mspr_aligned(x, 16) && mspr_aligned(out, 16), "fused_partial_rope: rows must be 16-byte aligned");
  hipStream_t st = (hipStream_t)stream;
  // The wide form where its blocks of positions are filled, in many small workgroups of four outer rows or more: 1008 MB of
  // float32 rows took 175, 169, 165, 160 us with 2048, 8192, 16384, 32768 workgroups (171 in the form below).
  // Past the caches from 24 M elements on: 31 M (3844 tokens of 64 x 128) gain by it, 17 M (517 of 64 x 512) in float32 lose
  // 4 %, for their rows still lie in the last-level cache.
  const int chunk_elems = dtype == MSPR_F32 ? 4 : 8;
  const int chunks = width / chunk_elems;
  if (width % chunk_elems == 0 && (chunks & (chunks - 1)) == 0 && chunks <= kThreads && seq_len >= kThreads / chunks) {
    const int log2 = __builtin_ctz(chunks);
    const int64_t pos_blocks = (seq_len + (kThreads >> log2) - 1) / (kThreads >> log2);
    int64_t slabs = (32768 + pos_blocks - 1) / pos_blocks;
    int64_t rows = (n_outer + slabs - 1) / slabs;
    if (rows < 4) rows = n_outer < 4 ? n_outer : 4;
    slabs = (n_outer + rows - 1) / rows;
    if (slabs <= 65535) {
      dim3 grid((unsigned)pos_blocks, (unsigned)slabs), block(kThreads);
      const bool stream_rows = n_outer * seq_len * width >= ((int64_t)24 << 20);
#define MSPR_ROPE_WIDE(DT, STREAM, STORE)                                                                                \
  partial_rope_wide_kernel<DT, STREAM, STORE><<<grid, block, 0, st>>>(x, (int)n_outer, (int)seq_len, log2, inv_freq,       \
                                                                      positions, offset, inverse, (int)rows, out)
      if (dtype == MSPR_F32) {
        if (stream_rows) MSPR_ROPE_WIDE(MSPR_F32, true, kStoreThrough);
        else MSPR_ROPE_WIDE(MSPR_F32, false, kStoreThrough);
      } else if (dtype == MSPR_F16) {
        if (stream_rows) MSPR_ROPE_WIDE(MSPR_F16, true, kStoreThrough);
        else MSPR_ROPE_WIDE(MSPR_F16, false, kStoreCached);
      } else {
        if (stream_rows) MSPR_ROPE_WIDE(MSPR_BF16, true, kStoreThrough);
        else MSPR_ROPE_WIDE(MSPR_BF16, false, kStoreCached);
      }
#undef MSPR_ROPE_WIDE
      MSPR_CHECK_LAUNCH("fused_partial_rope");
      return MSPR_OK;
    }
  }
  // slabs: enough workgroups to cover the chip, at least one quad per thread and pass
  const int quads = width / 4;
  int64_t rows_per_wg = (kThreads * 4 + quads - 1) / quads;  // about four passes of the thread block
  const int64_t want_wgs = 1024;
  const int64_t max_rows = (n_outer * seq_len + want_wgs - 1) / want_wgs;
  if (rows_per_wg > max_rows) rows_per_wg = max_rows;
  if (rows_per_wg < 1) rows_per_wg = 1;
  if (rows_per_wg > n_outer) rows_per_wg = n_outer;
  const int64_t slabs = (n_outer + rows_per_wg - 1) / rows_per_wg;
  MSPR_REQUIRE(slabs <= 65535, "fused_partial_rope: too many outer rows for one launch");
  dim3 grid((unsigned)seq_len, (unsigned)slabs), block(kThreads);
  if (dtype == MSPR_F32)
    partial_rope_kernel<MSPR_F32><<<grid, block, 0, st>>>(x, n_outer, seq_len, width, inv_freq, positions, offset,
                                                         inverse, (int)rows_per_wg, out);
  else if (dtype == MSPR_F16)
    partial_rope_kernel<MSPR_F16><<<grid, block, 0, st>>>(x, n_outer, seq_len, width, inv_freq, positions, offset,
                                                         inverse, (int)rows_per_wg, out);
  else
    partial_rope_kernel<MSPR_BF16><<<grid, block, 0, st>>>(x, n_outer, seq_len, width, inv_freq, positions, offset,
                                                          inverse, (int)rows_per_wg, out);
  MSPR_CHECK_LAUNCH("fused_partial_rope");
  return MSPR_OK;
}
