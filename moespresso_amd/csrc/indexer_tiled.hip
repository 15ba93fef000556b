// Prefill-side lightning-indexer scores over a chunk of tokens:
//   scores[b,t,c] = sum_h max(q[b,h,t] . comp[b,c], 0) * w[b,t,h],  -inf where c >= (pos0+t+1)/ratio
// Operands are staged as float16 (float32 inputs are rounded on load), products accumulate in float32
// on v_mfma_f32_32x32x16_f16 with heads = M and pool rows = N, so the relu / weight / head sum runs on
// the accumulator registers of one lane column per pool row.
//
// Workgroup = 4 waves = 4 consecutive tokens of one batch entry walking the same block of pool rows; the token's
// 64 x 128 query block stays in registers.
//
// Two forms of the product:
//  * Operands that came out of the indexer's QAT are, group of 32 by group of 32, values of the e2m1 lattice times a power
//    of two: exactly the operand format of v_mfma_scale_f32_32x32x64_f8f6f4 (fp4 with one e8m0 scale per 32), which
//    multiplies four times as many of them per cycle as the float16 form. Both operands are packed once per call into MFMA
//    operand order (pack_operands_kernel), where each value is checked by converting it back; the products are exact. Their
//    sums are exact too, and the scores those of the float16 form bit for bit, where the exponents of a dot product's four
//    group products lie within 9 of each other: in units of the smallest group's least product (a quarter, as lattice
//    values are multiples of one half) 32 products of at most 36 from each of four groups are at most 4 * 32 * 144 * 2^9 <
//    2^24 of them. (Rows of Gaussian values: within 2 per operand.) Groups further apart round in float32 in either form,
//    here once per 64 products and there once per 16: with group exponents drawn evenly from -13 .. 13 a dot product is off
//    by at most 0.9e-7 of the sum of its products' magnitudes, and by 2.0e-7 in the float16 form. With the
//    products this cheap the relu-weighted head sum on the vector units is the bound (two instructions per score and
//    head: 256 cycles of a wave's 32-row tile against 128 of the matrix pipe). Its tiles need no LDS and no barrier, so
//    the four waves drift apart and one wave's sums run under another's products.
//    3844 tokens x 7961 rows from position 28000: 24 us packing + 157 us (float16 form 633), vector units busy three
//    quarters of it; x 961 rows from position 0: 24 + 21 us (75); 517 tokens x 2053 rows: 7 + 14 us (46).
//  * Where a value is outside that lattice (a pool row, or a query of the workgroup's tokens) the same workgroup goes through
//    its rows in the float16 form, with pool tiles staged in LDS. (Three waves fit a SIMD with both forms in the kernel since
//    queries are rounded 32 heads at a time as they arrive; before, the float16 form was a launch of its own, 2 to 3 us of
//    every call: 517 x 2053 rows 22.0 -> 19.4, 255 x 1988 14.5 -> 12.1.) What the look at them costs operands that are not of
//    the format: 3844 float32 tokens x 961 rows 65 us in the float16 form alone, 74 with it; x 7961 rows 549 and 558; 517 x
//    2053 rows 45 and 48.
#include "common.h"
#include "profile.h"

namespace {

__device__ __forceinline__ uint32_t pack_h2(float a, float b) {
  typedef __attribute__((ext_vector_type(2))) _Float16 h2_t;
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{a, b}, h2_t));
}

// eight consecutive elements starting at element offset `off` as packed float16
template <int DT>
__device__ __forceinline__ u32x4_t load8_as_f16(const void* base, int64_t off) {
  if constexpr (DT == MSPR_F16) {
    return *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const uint16_t*>(base) + off);
  } else {
    const f32x4_t* p = reinterpret_cast<const f32x4_t*>(reinterpret_cast<const float*>(base) + off);
    const f32x4_t a = p[0], b = p[1];
    return u32x4_t{pack_h2(a.x, a.y), pack_h2(a.z, a.w), pack_h2(b.x, b.y), pack_h2(b.z, b.w)};
  }
}

// ---- fp4 form of the operands

typedef __attribute__((ext_vector_type(8))) int i32x8_t;

// A packed block: 64 rows of 128 (the heads of one token, or 64 pool rows) in MFMA operand order, [row / 32][k-step][lane]
// [16 bytes] with lane (n, g) holding columns 64 step + 32 g .. +31 of row n (+32), and one word of e8m0 scales per lane,
// byte 2 (row / 32) + step.
constexpr int kBlockRows = 64;
constexpr int kBlockCodeBytes = kBlockRows * 64;
constexpr int kBlockScaleBytes = 64 * 4;

// four consecutive elements, widened to float32
template <int DT>
__device__ __forceinline__ f32x4_t load4_as_f32(const void* base, int64_t off) {
  if constexpr (DT == MSPR_F16) {
    const u32x2_t x = *reinterpret_cast<const u32x2_t*>(reinterpret_cast<const uint16_t*>(base) + off);
    return f32x4_t{f16_bits_to_f32((uint16_t)(x.x & 0xFFFFu)), f16_bits_to_f32((uint16_t)(x.x >> 16)),
                   f16_bits_to_f32((uint16_t)(x.y & 0xFFFFu)), f16_bits_to_f32((uint16_t)(x.y >> 16))};
  } else {
    return *reinterpret_cast<const f32x4_t*>(reinterpret_cast<const float*>(base) + off);
  }
}

template <int M>
__device__ __forceinline__ uint32_t lane_xor_max(uint32_t v) {
  const uint32_t o = (uint32_t)__float_as_int(lane_xor<M>(__int_as_float((int)v)));
  return o > v ? o : v;
}

// The packed operands in the workspace.
struct PackedOperands {
  uint8_t* pool_codes;   // [batch][pool blocks] blocks
  uint8_t* q_codes;      // [batch][tokens] blocks
  uint8_t* pool_scales;
  uint8_t* q_scales;
  int32_t* pool_exact;   // one flag per block: every value is of the lattice
  int32_t* q_exact;
};

__host__ __device__ __forceinline__ int64_t pool_blocks(int64_t n_comp) { return (n_comp + kBlockRows - 1) / kBlockRows; }

inline size_t packed_bytes(int batch, int n_tokens, int64_t n_comp) {
  const size_t blocks = (size_t)batch * (pool_blocks(n_comp) + n_tokens);
  return blocks * (kBlockCodeBytes + kBlockScaleBytes + sizeof(int32_t));
}

inline PackedOperands packed_operands(void* workspace, int batch, int n_tokens, int64_t n_comp) {
  const int64_t pb = batch * pool_blocks(n_comp), qb = (int64_t)batch * n_tokens;
  PackedOperands o;
  o.pool_codes = reinterpret_cast<uint8_t*>(workspace);
  o.q_codes = o.pool_codes + pb * kBlockCodeBytes;
  o.pool_scales = o.q_codes + qb * kBlockCodeBytes;
  o.q_scales = o.pool_scales + pb * kBlockScaleBytes;
  o.pool_exact = reinterpret_cast<int32_t*>(o.q_scales + qb * kBlockScaleBytes);
  o.q_exact = o.pool_exact + pb;
  return o;
}

// Packs one block per workgroup. grid: (pool blocks + tokens, batch), 256 threads. Bound by the read of the queries, so all
// accesses are whole lines: eight neighbouring lanes read a group of 32 (16 bytes each in float32), find its largest
// magnitude by lane exchanges and convert four values each; the codes change to operand order in LDS.
//
// A group is stored times 2^e with the largest magnitude in [4, 8) * 2^e. (Lattice values times a power of two survive the
// shift to that range: doubling maps the lattice below 4 into itself.) A block is exact if every value converts back to
// itself and float16 could hold its groups exactly too.
template <int DT>
__global__ __launch_bounds__(256) void pack_operands_kernel(const void* __restrict__ q, const void* __restrict__ comp,
                                                            int n_heads, int n_tokens, int64_t n_comp, PackedOperands out) {
  __shared__ __attribute__((aligned(16))) uint16_t codes[kBlockCodeBytes / 2];
  __shared__ __attribute__((aligned(16))) uint8_t scales[kBlockScaleBytes];
  const int tid = threadIdx.x;
  const int64_t n_pool = pool_blocks(n_comp), b = blockIdx.y;
  const bool is_pool = (int64_t)blockIdx.x < n_pool;
  const int64_t x = is_pool ? blockIdx.x : blockIdx.x - n_pool;  // pool block, or token
  const void* src = is_pool ? comp : q;
  const int64_t row0 = is_pool ? b * n_comp + x * kBlockRows : b * n_heads * n_tokens + x;
  const int64_t row_step = is_pool ? 1 : n_tokens;
  const int64_t left = is_pool ? n_comp - x * kBlockRows : n_heads;
  const int n_rows = left < kBlockRows ? (int)left : kBlockRows;
  const int col = (tid & 31) * 4;  // 32 lanes a row: eight rows per pass of the workgroup
  auto load = [&](int i) -> f32x4_t {
    // (Past the block the last row again: under a condition a load is waited for before the next, 28.4 us and 26.9 for 3844
    // tokens.)
    const int r = 8 * i + (tid >> 5);
    return load4_as_f32<DT>(src, (row0 + (r < n_rows ? r : n_rows - 1) * row_step) * 128 + col);
  };
  auto pack = [&](int i, f32x4_t v) -> bool {
    const int r = 8 * i + (tid >> 5);
    if (r >= n_rows) v = f32x4_t{0.f, 0.f, 0.f, 0.f};
    uint32_t top = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const uint32_t a = __float_as_uint(v[j]) & 0x7FFFFFFFu;
      top = a > top ? a : top;
    }
    top = lane_xor_max<4>(lane_xor_max<2>(lane_xor_max<1>(top)));
    const int e = top == 0u ? 0 : (int)(top >> 23) - 127 - 2;
    const float scale = __uint_as_float((uint32_t)(e + 127) << 23);
    uint32_t c = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(0u, v.x, v.y, scale, 0);
    c = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(c, v.z, v.w, scale, 1);
    const f32x2_t b0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c, scale, 0), b1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c, scale, 1);
    const int group = (tid & 31) >> 3, k = tid & 7;
    const int lane = (r & 31) + 32 * (group & 1), part = 2 * (r >> 5) + (group >> 1);
    codes[(part * 64 + lane) * 8 + k] = (uint16_t)c;
    if (k == 0) scales[lane * 4 + part] = (uint8_t)(e + 127);
    return e >= -13 && e <= 13 && b0.x == v.x && b0.y == v.y && b1.x == v.z && b1.y == v.w;
  };
  const int64_t block = is_pool ? b * n_pool + x : b * n_tokens + x;
  int32_t* flag = (is_pool ? out.pool_exact : out.q_exact) + block;
  // The first eight rows decide whether the rest is read at all: values that did not come out of the QAT end here.
  bool exact = pack(0, load(0));
  if (!__syncthreads_and(exact)) {
    if (tid == 0) *flag = 0;
    return;
  }
  f32x4_t v[8];
#pragma unroll
  for (int i = 1; i < 8; i++) v[i] = load(i);
#pragma unroll
  for (int i = 1; i < 8; i++) exact = pack(i, v[i]) && exact;
  const int all = __syncthreads_and(exact);
  uint8_t* cp = (is_pool ? out.pool_codes : out.q_codes) + block * kBlockCodeBytes;
  uint8_t* sp = (is_pool ? out.pool_scales : out.q_scales) + block * kBlockScaleBytes;
  reinterpret_cast<u32x4_t*>(cp)[tid] = reinterpret_cast<const u32x4_t*>(codes)[tid];
  if (tid < 64) reinterpret_cast<uint32_t*>(sp)[tid] = reinterpret_cast<const uint32_t*>(scales)[tid];
  if (tid == 0) *flag = all;
}

// Whether all operands of the workgroup (the whole pool of its batch entry, its four tokens) are exact. Every thread makes
// one and asks it once; the flags are requested in between, ahead of what the caller loads meanwhile.
struct OperandsExact {
  const int32_t* pool;
  int64_t n;
  int32_t pool_flag, q_flag;

  __device__ __forceinline__ OperandsExact(const PackedOperands& o, int n_tokens, int64_t n_comp) {
    n = pool_blocks(n_comp);
    pool = o.pool_exact + blockIdx.z * n;
    const int t = blockIdx.y * 4 + (threadIdx.x & 3);
    pool_flag = pool[(int64_t)threadIdx.x < n ? threadIdx.x : 0];
    q_flag = o.q_exact[(int64_t)blockIdx.z * n_tokens + (t < n_tokens ? t : n_tokens - 1)];
  }
  __device__ __forceinline__ bool all() const {
    bool exact = pool_flag != 0 && q_flag != 0;
    for (int64_t i = threadIdx.x + 256; i < n; i += 256) exact = exact && pool[i] != 0;
    return __syncthreads_and(exact);
  }
};

// max(x, 0) of a number that is no NaN, as one integer maximum (fmaxf costs a second instruction that quiets NaNs)
__device__ __forceinline__ float relu_finite(float x) {
  const int b = __float_as_int(x);
  return __int_as_float(b > 0 ? b : 0);
}

// What one wave of a score workgroup works on: its token and the workgroup's block of pool rows.
struct ScoreJob {
  int lane, n, g;  // lane; operand row (head or pool row) and half
  int b, t;        // batch entry, token (the last one where the chunk ends inside the workgroup: t_live is false)
  bool t_live;
  int64_t row_begin, row_end, visible;
  int n_live;   // tiles of the block that hold a row visible to the token
  int n_fetch;  // the same for the workgroup's last token, which sees the most
  float* out_row;

  __device__ __forceinline__ ScoreJob(int n_tokens, int64_t n_comp, uint32_t pos0, uint32_t ratio, int rows_per_block,
                                      float* scores) {
    lane = threadIdx.x & 63;
    n = lane & 31;
    g = lane >> 5;
    b = blockIdx.z;
    t = blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    t_live = t < n_tokens;
    if (!t_live) t = n_tokens - 1;
    row_begin = (int64_t)blockIdx.x * rows_per_block;
    row_end = row_begin + rows_per_block;
    if (row_end > n_comp) row_end = n_comp;
    auto visible_of = [&](int tok) -> int64_t {
      const uint32_t qpos1 = pos0 + (uint32_t)tok + 1u;
      const int64_t v = ratio == 0u ? n_comp : (int64_t)(qpos1 / ratio);
      return v < n_comp ? v : n_comp;
    };
    auto live_tiles = [&](int64_t vis) -> int {
      const int64_t live_end = vis < row_end ? vis : row_end;
      return live_end > row_begin ? (int)((live_end - row_begin + 31) / 32) : 0;
    };
    visible = visible_of(t);
    n_live = live_tiles(visible);
    int t_last = blockIdx.y * 4 + 3;
    if (t_last > n_tokens - 1) t_last = n_tokens - 1;
    n_fetch = live_tiles(visible_of(t_last));
    out_row = scores + ((int64_t)b * n_tokens + t) * n_comp;
  }

  // rows of the block behind the `n_done` tiles that were multiplied: not visible to this token
  __device__ __forceinline__ void mask_rest(int n_done) const {
    if (!t_live) return;
    for (int64_t c = row_begin + (int64_t)n_done * 32 + lane; c < row_end; c += 64) out_row[c] = -__builtin_inff();
  }

  // weights of the heads this lane's accumulator registers hold: head = 32 hb + 8 (i/4) + 4 g + i%4
  __device__ __forceinline__ void head_weights(const float* __restrict__ w, int n_tokens, int n_heads,
                                               float (&wv)[2][16]) const {
    const float* w_row = w + ((int64_t)b * n_tokens + t) * n_heads;
    if (n_heads == 64 && (reinterpret_cast<uintptr_t>(w) & 15u) == 0) {  // (four consecutive heads per load)
#pragma unroll
      for (int hb = 0; hb < 2; hb++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const f32x4_t v = *reinterpret_cast<const f32x4_t*>(w_row + 32 * hb + 8 * j + 4 * g);
          wv[hb][4 * j] = v.x;
          wv[hb][4 * j + 1] = v.y;
          wv[hb][4 * j + 2] = v.z;
          wv[hb][4 * j + 3] = v.w;
        }
    } else {
#pragma unroll
      for (int hb = 0; hb < 2; hb++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
          const int head = 32 * hb + 8 * (i / 4) + 4 * g + (i % 4);
          wv[hb][i] = head < n_heads ? w_row[head] : 0.0f;
        }
    }
  }
};

// A workgroup = 4 waves = 4 consecutive tokens walks `rows_per_block` pool rows (a multiple of 64) in tiles of 32. Float16
// form:
// A tile is fetched once per workgroup (every thread 32 bytes of it, rounded to float16) into one of two LDS buffers,
// a tile ahead of its use, and the four waves read their B operands from there: fetched by each wave for itself, the
// 16-byte pieces of 32 rows keep a CU's address path busier than its matrix pipes. Rows past a token's visible
// prefix score -inf whatever the products are, so a wave multiplies only the tiles that hold a row it sees.
constexpr int kTilePitch = 272;  // bytes between rows of a tile in LDS: 256 + 16, operand reads of 32 rows x 2 pieces
                                 // and the 16-byte writes of two rows at a time both without bank conflicts

template <int DT>
__device__ __forceinline__ void scores_f16(const ScoreJob& j, const void* __restrict__ q, const float* __restrict__ w,
                                           const void* __restrict__ comp, int n_heads, int n_tokens, int64_t n_comp,
                                           unsigned char (&tile_lds)[2][32 * kTilePitch]) {
  const int tid = threadIdx.x, n = j.n, g = j.g, b = j.b, t = j.t;
  const int n_live = j.n_live, n_fetch = j.n_fetch;
  const int64_t row_begin = j.row_begin;

  if (n_fetch > 0) {  // (the same in every wave of the workgroup: the barriers below are met by all)
    const void* comp_b =
        DT == MSPR_F16 ? static_cast<const void*>(reinterpret_cast<const uint16_t*>(comp) + (int64_t)b * n_comp * 128)
                       : static_cast<const void*>(reinterpret_cast<const float*>(comp) + (int64_t)b * n_comp * 128);
    // this thread's share of a tile: row tid / 8, columns [16 (tid % 8), +16)
    const int f_row = tid >> 3, f_col = (tid & 7) * 16;
    auto fetch = [&](int64_t r0, u32x4_t (&st)[2]) {
      int64_t row = r0 + f_row;
      if (row >= n_comp) row = n_comp - 1;
      st[0] = load8_as_f16<DT>(comp_b, row * 128 + f_col);
      st[1] = load8_as_f16<DT>(comp_b, row * 128 + f_col + 8);
    };
    auto stash = [&](int buf, const u32x4_t (&st)[2]) {
      unsigned char* p = tile_lds[buf] + f_row * kTilePitch + f_col * 2;
      *reinterpret_cast<u32x4_t*>(p) = st[0];
      *reinterpret_cast<u32x4_t*>(p + 16) = st[1];
    };
    u32x4_t st[2];
    fetch(row_begin, st);  // (in flight while the query block and the weights arrive)

    // A operand: q[b, head, t, 16 s + 8 g .. +7] for head = n (+32), zero rows past n_heads
    u32x4_t qa[2][8];
#pragma unroll
    for (int hb = 0; hb < 2; hb++) {
      const int head = 32 * hb + n;
      const bool live = head < n_heads;
      const int64_t off = (((int64_t)b * n_heads + (live ? head : 0)) * n_tokens + t) * 128 + 8 * g;
#pragma unroll
      for (int s = 0; s < 8; s++) {
        u32x4_t v = load8_as_f16<DT>(q, off + 16 * s);
        qa[hb][s] = live ? v : u32x4_t{0, 0, 0, 0};
      }
      // (rounded here: the rest of the block does not fit the registers in float32)
#pragma unroll
      for (int s = 0; s < 8; s++) asm volatile("" : "+v"(qa[hb][s]));
    }
    float wv[2][16];
    j.head_weights(w, n_tokens, n_heads, wv);
    stash(0, st);
    __syncthreads();

    for (int i = 0; i < n_fetch; i++) {
      if (i + 1 < n_fetch) fetch(row_begin + 32 * (int64_t)(i + 1), st);
      if (i < n_live) {
        // B operand: lane (n, g) holds comp[row r0 + n][16 s + 8 g .. +7] for k-step s
        const unsigned char* kt = tile_lds[i & 1] + n * kTilePitch + 16 * g;
        f32x16_t acc0 = {0}, acc1 = {0};
#pragma unroll
        for (int s = 0; s < 8; s++) {
          const u32x4_t kb = *reinterpret_cast<const u32x4_t*>(kt + 32 * s);
          acc0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, qa[0][s]),
                                                        __builtin_bit_cast(f16x8_t, kb), acc0, 0, 0, 0);
          acc1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, qa[1][s]),
                                                        __builtin_bit_cast(f16x8_t, kb), acc1, 0, 0, 0);
        }
        float sum = 0.0f;
#pragma unroll
        for (int k = 0; k < 16; k++) {
          sum += fmaxf(acc0[k], 0.0f) * wv[0][k];
          sum += fmaxf(acc1[k], 0.0f) * wv[1][k];
        }
        sum += __shfl_xor(sum, 32, MSPR_WAVE);
        const int64_t c = row_begin + 32 * (int64_t)i + n;
        if (j.t_live && g == 0 && c < j.row_end) j.out_row[c] = c < j.visible ? sum : -__builtin_inff();
      }
      if (i + 1 < n_fetch) stash((i + 1) & 1, st);
      __syncthreads();  // tile i+1 written by every thread; tile i read by every wave
    }
  }
  j.mask_rest(n_live);
}

template <int DT>
__global__ __launch_bounds__(256, 2) void scores_tiled_kernel(const void* __restrict__ q, const float* __restrict__ w,
                                                           const void* __restrict__ comp, int n_heads, int n_tokens,
                                                           int64_t n_comp, uint32_t pos0, uint32_t ratio,
                                                           int rows_per_block, float* __restrict__ scores) {
  __shared__ __attribute__((aligned(16))) unsigned char tile_lds[2][32 * kTilePitch];
  scores_f16<DT>(ScoreJob(n_tokens, n_comp, pos0, ratio, rows_per_block, scores), q, w, comp, n_heads, n_tokens, n_comp,
                 tile_lds);
}

// fp4 form, or the float16 form where the operands are not of the format. grid: (row blocks, token blocks, batch); a wave
// walks its rows in pairs of tiles, one packed block at a time.
__global__ __launch_bounds__(256, 3) void scores_fp4_kernel(const float* __restrict__ w, int n_heads, int n_tokens,
                                                            int64_t n_comp, uint32_t pos0, uint32_t ratio,
                                                            int rows_per_block, float* __restrict__ scores,
                                                            PackedOperands ops, const void* __restrict__ q,
                                                            const void* __restrict__ comp, int dtype) {
  __shared__ __attribute__((aligned(16))) unsigned char tile_lds[2][32 * kTilePitch];
  const ScoreJob j(n_tokens, n_comp, pos0, ratio, rows_per_block, scores);
  if (j.n_fetch == 0) {  // no row of the block is visible to any of the four tokens, whatever the operands are
    j.mask_rest(0);
    return;
  }
  const OperandsExact exact(ops, n_tokens, n_comp);  // (first, so that a workgroup without work waits for nothing else)
  const int n_pairs = (j.n_live + 1) / 2;
  const int64_t block0 = j.b * pool_blocks(n_comp) + j.row_begin / kBlockRows;
  const u32x4_t* cp = reinterpret_cast<const u32x4_t*>(ops.pool_codes + block0 * kBlockCodeBytes) + j.lane;
  const uint32_t* sp = reinterpret_cast<const uint32_t*>(ops.pool_scales + block0 * kBlockScaleBytes) + j.lane;
  struct Rows {
    u32x4_t c[2][2];
    uint32_t s;
  } even, odd;
  auto fetch = [&](Rows& k, int pair) {
    if (pair >= n_pairs) pair = n_pairs - 1;  // (a last fetch that nothing uses)
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int s = 0; s < 2; s++) k.c[u][s] = cp[pair * (kBlockCodeBytes / 16) + (2 * u + s) * 64];
    k.s = sp[pair * 64];
  };
  if (n_pairs > 0) fetch(even, 0);
  u32x4_t qa[2][2];
  const int64_t token = (int64_t)j.b * n_tokens + j.t;
  const u32x4_t* qp = reinterpret_cast<const u32x4_t*>(ops.q_codes + token * kBlockCodeBytes) + j.lane;
#pragma unroll
  for (int hb = 0; hb < 2; hb++)
#pragma unroll
    for (int s = 0; s < 2; s++) qa[hb][s] = qp[(2 * hb + s) * 64];
  const uint32_t qs = reinterpret_cast<const uint32_t*>(ops.q_scales + token * kBlockScaleBytes)[j.lane];
  float wv[2][16];
  j.head_weights(w, n_tokens, n_heads, wv);
  if (!exact.all()) {
    if (dtype == MSPR_F16) scores_f16<MSPR_F16>(j, q, w, comp, n_heads, n_tokens, n_comp, tile_lds);
    else scores_f16<MSPR_F32>(j, q, w, comp, n_heads, n_tokens, n_comp, tile_lds);
    return;
  }

  float* out = j.out_row + j.row_begin + j.lane;
  int left = (int)(j.row_end - j.row_begin) - j.lane, seen = (int)(j.visible - j.row_begin) - j.lane;
  if (!j.t_live) left = 0;
  auto step = [&](const Rows& k, int pair) {
    f32x16_t acc[2][2];
#define MSPR_FP4_STEP(u, hb, st)                                                                                   \
  acc[u][hb] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(                                                    \
      i32x8_t{(int)qa[hb][st].x, (int)qa[hb][st].y, (int)qa[hb][st].z, (int)qa[hb][st].w, 0, 0, 0, 0},             \
      i32x8_t{(int)k.c[u][st].x, (int)k.c[u][st].y, (int)k.c[u][st].z, (int)k.c[u][st].w, 0, 0, 0, 0},             \
      st == 0 ? f32x16_t{0} : acc[u][hb], 4, 4, 2 * hb + st, (int)qs, 2 * u + st, (int)k.s)
    MSPR_FP4_STEP(0, 0, 0);
    MSPR_FP4_STEP(0, 1, 0);
    MSPR_FP4_STEP(0, 0, 1);
    MSPR_FP4_STEP(0, 1, 1);
    MSPR_FP4_STEP(1, 0, 0);
    MSPR_FP4_STEP(1, 1, 0);
    MSPR_FP4_STEP(1, 0, 1);
    MSPR_FP4_STEP(1, 1, 1);
#undef MSPR_FP4_STEP
    float sum[2] = {0.0f, 0.0f};
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int i = 0; i < 16; i++) {
        sum[u] += relu_finite(acc[u][0][i]) * wv[0][i];
        sum[u] += relu_finite(acc[u][1][i]) * wv[1][i];
      }
    // the exchange adds the two halves of a tile's heads and leaves the first tile's scores in the lower half-wave, the
    // second's in the upper one: 256 bytes are stored at once
    half_wave_exchange(sum[0], sum[1]);
    const int c = 64 * pair;
    if (c < left) out[c] = c < seen ? sum[0] + sum[1] : -__builtin_inff();
  };
  for (int i = 0; i < n_pairs; i += 2) {
    fetch(odd, i + 1);
    __builtin_amdgcn_sched_barrier(0);  // (requested before the products it hides behind, not after them)
    step(even, i);
    if (i + 1 >= n_pairs) break;
    fetch(even, i + 2);
    __builtin_amdgcn_sched_barrier(0);
    step(odd, i + 1);
  }
  j.mask_rest(2 * n_pairs);
}

}  // namespace

extern "C" size_t mspr_indexer_scores_tiled_live_workspace_bytes(int batch, int n_heads, int n_tokens, int64_t n_comp) {
  if (batch < 1 || n_heads < 1 || n_tokens < 1 || n_comp < 1) return 0;
  return packed_bytes(batch, n_tokens, n_comp);
}

extern "C" int mspr_indexer_scores_tiled_live_ws(const void* q, const float* weights, const void* index_comp, int dtype,
                                                 int batch, int n_heads, int n_tokens, int64_t n_comp, int64_t pos0,
                                                 int ratio, float* scores, void* workspace, size_t workspace_bytes,
                                                 void* stream) {
  MSPR_REQUIRE(q && weights && index_comp && scores, "indexer_scores_tiled_live: null pointer");
  MSPR_REQUIRE(dtype == MSPR_F32 || dtype == MSPR_F16,
               "indexer_scores_tiled_live: q and index_comp must both be float32 or both be float16");
  MSPR_REQUIRE(batch >= 1 && n_tokens >= 1, "indexer_scores_tiled_live: q must contain at least one batch and token");
  MSPR_REQUIRE(n_heads >= 1 && n_heads <= 64, "indexer_scores_tiled_live: between 1 and 64 heads");
  MSPR_REQUIRE(n_comp >= 1, "indexer_scores_tiled_live: index_comp must contain at least one compressed row");
  MSPR_REQUIRE(pos0 >= 0 && ratio >= 0 && pos0 + n_tokens < ((int64_t)1 << 31) && batch <= 65535,
               "indexer_scores_tiled_live: bad size argument");
  MSPR_REQUIRE(mspr_aligned(q, 16) && mspr_aligned(index_comp, 16),
               "indexer_scores_tiled_live: pointers must be 16-byte aligned");
  MSPR_REQUIRE(!workspace || (workspace_bytes >= packed_bytes(batch, n_tokens, n_comp) && mspr_aligned(workspace, 16)),
               "indexer_scores_tiled_live: workspace of %zu bytes (16-byte aligned) needed, %zu given",
               packed_bytes(batch, n_tokens, n_comp), workspace_bytes);
  // Four tokens per workgroup; the pool rows are split over several workgroups only as far as it takes to have
  // `want` workgroups, and no finer than `least` pairs of tiles.
  const int64_t tok_blocks = (n_tokens + 3) / 4;
  const int64_t row_pairs = (n_comp + 63) / 64;
  auto rows_per_workgroup = [&](int64_t want, int64_t least) -> int64_t {
    int64_t blocks = (want + tok_blocks * batch - 1) / (tok_blocks * batch);
    if (blocks > row_pairs / least) blocks = row_pairs / least;
    if (blocks < 1) blocks = 1;
    return (row_pairs + blocks - 1) / blocks * 64;
  };
  hipStream_t st = (hipStream_t)stream;
  dim3 block(256);
  PackedOperands packed = {};
  // The fp4 form is a launch more, some 3 us and what packing takes, which cheaper products have to earn. The float16 form runs
  // in rounds of 256 pieces (64 rows for four tokens, one to a CU) of 4.3 us with float32 operands, which it rounds as it loads
  // them, and of 2.4 us with float16 ones. float32: from the second round on, unless a token's 64 queries are packed for no more
  // than 64 rows. float16: from the fifth full round on, and behind it where the packed blocks are many. us without and with it,
  // float32: 64 tokens x 1000 rows (256 pieces) 7.2 and 8.5, 66 x 1000 11.4 and 8.6, 400 x 1000 25.5 and 11.5, 530 x 128 13.2 and
  // 9.3, 3844 x 100 26.2 and 29.7, 1 x 20000 11.5 and 9.9, 2000 x 33 13.2 and 17.2, 4097 x 33 24.8 and 30.8. float16: 256 x 1000
  // (1024) 9.9 and 10.0, 270 x 1000 12.4 and 10.9, 400 x 1000 17.8 and 11.6, 520 x 500 12.4 and 12.1, 1300 x 256 13.5 and 15.4,
  // 1562 x 256 17.1 and 15.8, 3844 x 128 19.7 and 25.0, 3844 x 256 26.3 and 27.4, 1 x 120000 15.0 and 18.4. Operands that are not
  // of the format, and that the caller does not name as such, pay for being looked at: 90 x 1000 float32 11.4 and 16.3, 131 x
  // 1000 15.9 and 16.6; 330 x 1000 float16 13.9 and 17.2, 400 x 1000 18.0 and 17.6.
  const int64_t packed_blocks = (row_pairs + n_tokens) * batch, token_pairs = row_pairs * n_tokens * batch;
  const bool fp4_pays = dtype == MSPR_F32 ? row_pairs * tok_blocks * batch > 256 && row_pairs > 1
                                          : token_pairs > 4 * 1024 && token_pairs > 3072 + 2 * packed_blocks;
  if (workspace && fp4_pays) {
    packed = packed_operands(workspace, batch, n_tokens, n_comp);
    const int64_t blocks = pool_blocks(n_comp) + n_tokens;
    MSPR_REQUIRE(blocks < ((int64_t)1 << 31) && tok_blocks <= 65535 && n_comp < ((int64_t)1 << 31),
                 "indexer_scores_tiled_live: grid too large");
    dim3 pgrid((unsigned)blocks, (unsigned)batch);
    if (dtype == MSPR_F16)
      pack_operands_kernel<MSPR_F16><<<pgrid, block, 0, st>>>(q, index_comp, n_heads, n_tokens, n_comp, packed);
    else
      pack_operands_kernel<MSPR_F32><<<pgrid, block, 0, st>>>(q, index_comp, n_heads, n_tokens, n_comp, packed);
    // A workgroup's start (operands, flags: some 3 us) has to be carried by its tiles: at least 16 pairs of them, or 8 where
    // the chip is not full otherwise, or 4 where there are not two workgroups to a CU even so. Three rounds of workgroups level
    // the last one: 3844 tokens x 7961 rows took 164, 160, 157, 168 us with 1, 2, 3, 4 row blocks, x 961 rows from position 0
    // took 21, 25, 31 us with 1, 2, 4; 517 tokens x 2053 rows 15.5 us with 2 and 13.7 us with 4. At least 8 and 4 pairs, whole
    // calls: 96 x 2000 10.9 and 9.3 (random operands 23.7 and 16.9), 64 x 4000 11.4 and 9.7, 300 x 600 12.2 and 10.3, 1200 x 500
    // 17.9 and 17.0, 528 x 1000 14.6 and 13.7. Where 8 leave just under a workgroup to a CU, either: 928 x 500 float32 13.7 and
    // 14.4, 928 x 600 float16 15.4 and 14.8. From 512 on 8: 517 x 2053 19.4 and 20.2.
    int64_t rows = rows_per_workgroup(2304, 16);
    auto workgroups = [&]() -> int64_t { return (n_comp + rows - 1) / rows * tok_blocks * batch; };
    if (workgroups() < 768) rows = rows_per_workgroup(768, 8);
    if (workgroups() < 512) rows = rows_per_workgroup(768, 4);
    dim3 grid((unsigned)((n_comp + rows - 1) / rows), (unsigned)tok_blocks, (unsigned)batch);
    scores_fp4_kernel<<<grid, block, 0, st>>>(weights, n_heads, n_tokens, n_comp, (uint32_t)pos0, (uint32_t)ratio,
                                              (int)rows, scores, packed, q, index_comp, dtype);
    MSPR_CHECK_LAUNCH("indexer_scores_tiled_live (fp4)");
    return MSPR_OK;
  }
  // float16 form: three rounds of workgroups where each has sixteen pairs of tiles, else about one (every workgroup fetches
  // its tokens' query blocks anew). 3844 tokens x 7961 rows one round 619 us, three 559.
  int64_t rows = rows_per_workgroup(2304, 16);
  if ((n_comp + rows - 1) / rows * tok_blocks * batch < 768) rows = rows_per_workgroup(768, 1);
  const int64_t row_blocks = (n_comp + rows - 1) / rows;
  MSPR_REQUIRE(row_blocks < ((int64_t)1 << 31) && tok_blocks <= 65535 && rows < ((int64_t)1 << 31),
               "indexer_scores_tiled_live: grid too large");
  dim3 grid((unsigned)row_blocks, (unsigned)tok_blocks, (unsigned)batch);
  if (dtype == MSPR_F16)
    scores_tiled_kernel<MSPR_F16><<<grid, block, 0, st>>>(q, weights, index_comp, n_heads, n_tokens, n_comp, (uint32_t)pos0,
                                                          (uint32_t)ratio, (int)rows, scores);
  else
    scores_tiled_kernel<MSPR_F32><<<grid, block, 0, st>>>(q, weights, index_comp, n_heads, n_tokens, n_comp, (uint32_t)pos0,
                                                          (uint32_t)ratio, (int)rows, scores);
  MSPR_CHECK_LAUNCH("indexer_scores_tiled_live");
  return MSPR_OK;
}

extern "C" int mspr_indexer_scores_tiled_live(const void* q, const float* weights, const void* index_comp, int dtype,
                                              int batch, int n_heads, int n_tokens, int64_t n_comp, int64_t pos0,
                                              int ratio, float* scores, void* stream) {
  return mspr_indexer_scores_tiled_live_ws(q, weights, index_comp, dtype, batch, n_heads, n_tokens, n_comp, pos0, ratio,
                                           scores, nullptr, 0, stream);
}
