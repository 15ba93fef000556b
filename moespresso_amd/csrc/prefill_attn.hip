// Indexed prefill attention: every token of a chunk attends the rows of its sliding window (a ring) and pool rows that its
// own id list names. K == V, 512 wide float16 rows shared by all heads; a per-head sink joins the denominator.
//
// Visit rules (reference: indexed_attention_kernel.py:120-173 of src/moespresso/runtime/deepseek_v4): ring rows for positions
// [max(first_raw, pos+1-window), min(pos, last)], then the ids in order; a negative id is skipped and the first id at or
// behind min((pos+1)/ratio, n_pool) ends the walk.
//
// Split: a workgroup is four waves and owns one token and 64 heads; a wave owns 16 of the heads outright: the 16 x 512 query
// block (64 registers), the whole 512-wide output (128 registers) and the softmax state of its heads. Nothing but the row
// tiles is shared between the waves, so a tile costs one barrier: tiles of 32 rows lie in two LDS buffers, the copies of
// tile t+1 (asynchronous, one 1 KB row per instruction, its address scalar) are issued behind the barrier of tile t and land
// under its arithmetic. S^T = K.Q^T leaves a wave's weights in the registers that O^T += V^T.P^T wants as its B operand
// (the key order inside a tile is free as long as V^T uses the same), V^T comes out of the row-major tile by transpose reads.
//
// Two such workgroups share a CU (80 KB of LDS and 256 registers a lane each) and drift apart: one multiplies while the
// other waits for its barrier, its ids, or takes its exponentials. The price is LDS traffic: each wave reads the whole tile
// for both products, 256 KB per tile and workgroup, which bounds the kernel: the two products alone need 2800 cycles of a
// pair of workgroups' tiles, the matrix pipes 2050, and it takes 3100 (2.15 GHz).
//
// 3844 tokens, 64 heads, 128 + 512 rows each: from position 28000 426 us with float32 queries (before, with eight waves of
// a persistent workgroup on one token and the queries rounded to half in a pass of their own: 620 + 130), from position 0
// 324 us (542); 517 tokens 62 us (121). Without the tile copies 355 / 295 us, without the stores 360 / 276, with neither
// 303 / 240, which is the products and the softmax. Measured and not kept: one wave for 128 output columns of all heads
// (V^T read once per workgroup, weights exchanged through LDS behind a second barrier) 500 / 397; persistent workgroups
// that request the next token's ids, rows and queries under the last tile 471 / 351 with the stores as they were (464 / 361
// without).
#include "prefill_attn.h"
#include "profile.h"

namespace {

constexpr int kTile = 32;
constexpr int kThreads = 256;
constexpr int kD = 512;
constexpr int kPitch = kD * 2 + 32;  // bytes between rows in LDS: both read patterns run fastest at this distance
constexpr int kTileBytes = kTile * kPitch;
constexpr int kOffIds = 2 * kTileBytes;
constexpr int kLdsBytes = 80 * 1024;                       // half of a CU's
constexpr int kMaxIds = (kLdsBytes - kOffIds - 64) / 4 / 64 * 64;
constexpr int kOffStop = kOffIds + kMaxIds * 4;
static_assert(kOffStop + 4 <= kLdsBytes, "LDS map");
constexpr int kQSteps = kD / 32;
constexpr int kOutPitch = 256 + 4;  // floats between rows of the output staging: 16 heads' stores fall on 16 bank groups
static_assert(4 * 16 * kOutPitch * 4 <= 2 * kTileBytes, "output staging lies in the tile buffers");
constexpr int kMaxRanges = 8;
constexpr int kRound = 512;  // units at work at once: two to a CU
constexpr int kAheadK = 8, kAheadV = 6;  // operand reads in flight (6/4 measures the same, 10/8 9 % slower)

__device__ __attribute__((aligned(16))) const unsigned char g_prefill_zero_row[kD * 2] = {0};

__device__ __forceinline__ f32x4_t mfma16(u32x4_t a, u32x4_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

__device__ __forceinline__ uint32_t pack_h2(float a, float b) {
  typedef __attribute__((ext_vector_type(2))) _Float16 h2_t;
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{a, b}, h2_t));
}

// One 1 KB row to LDS: lane l's 16 bytes go to lds_base + 16 l. Through asm so that the compiler does not drain it in front
// of LDS reads; the tile loop waits for all copies of a tile at its barrier. (An instruction has to stand between a scalar
// write of M0 and the copy that takes its LDS address from it; the compiler, which sees to that elsewhere, does not look
// inside an asm statement.)
__device__ __forceinline__ void async_row(uint64_t row, uint32_t lane_off, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lane_off), "s"(row), "s"(lds_base)
               : "memory", "m0");
}

// CUT: the launch has units that are cut into key ranges (compiled in, the choice cost whole units 3 %).
// (Plain arguments first: what the first copies and the ids of up to 64 heads of one sequence take comes in registers with the
// wave, and the struct is loaded meanwhile: it was loaded in three dependent steps with three software divisions between. One
// token behind 28000 rows 22.1 -> 21.6 us with its merge, 255 tokens 43.8 -> 43.5; full rounds, which power bounds, are as they
// were. With how the units are cut among the plain words, and the block 136 bytes instead of 224, whole calls of 1, 17 and 60
// tokens 11.7 -> 11.5, 20.0 -> 19.9, 23.7 -> 23.5; calls that are not cut the same within 0.3 %. cut: split_units, and ranges from bit 16 on; inv_ranges: mspr_inverse(ranges).)
template <int QDT, bool CUT>
__global__ __launch_bounds__(kThreads, 2) void indexed_prefill_kernel(const void* win, const int32_t* idx, int units,
                                                                      int n_tokens, int n_hblk, uint32_t pos0,
                                                                      uint32_t window, uint32_t n_raw, int raw_start,
                                                                      int n_idx, uint32_t cut, uint32_t inv_ranges,
                                                                      IndexedPrefillRest a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  int* ids = reinterpret_cast<int*>(lds + kOffIds);
  int* stop_sh = reinterpret_cast<int*>(lds + kOffStop);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c16 = lane & 15;  // head of the wave (MFMA column), or row of an operand block
  const int kg = lane >> 4;

  // The tokens with the most rows (the last ones, at the start of a context) are started first.
  // The first split_units units, a part-filled last round, are cut into that many key ranges each and come last.
  const int split_units = (int)(cut & 0xFFFFu), ranges = (int)(cut >> 16);
  int unit = units - 1 - (int)blockIdx.x, range = 0;
  bool split = false;
  if constexpr (CUT) {
    const int whole = units - split_units;
    split = (int)blockIdx.x >= whole;
    const int i = (int)blockIdx.x - whole;
    unit = split ? mspr_div(i, ranges, inv_ranges) : split_units - 1 - i;
    range = split ? i - unit * ranges : 0;
  }
  // (real divisions, but in branches that 64 heads of one sequence pass by: reciprocals of both in the struct were loaded, and
  // waited for, in front of the branches)
  const int seq = n_hblk == 1 ? unit : unit / n_hblk;
  const int hb = unit - seq * n_hblk;
  const int b = seq < n_tokens ? 0 : seq / n_tokens;
  const int t = seq - b * n_tokens;

  // window rows and visible pool prefix, in the unsigned 32-bit arithmetic of the reference kernel
  const uint32_t qpos = pos0 + (uint32_t)t;
  const uint32_t last_pos = pos0 + (uint32_t)n_tokens - 1u;
  const uint32_t first_raw_pos = last_pos + 1u - n_raw;
  const uint32_t window_first = (window != 0u && qpos + 1u > window) ? qpos + 1u - window : 0u;
  const uint32_t first = first_raw_pos > window_first ? first_raw_pos : window_first;
  const uint32_t last = qpos < last_pos ? qpos : last_pos;
  const int n_win = first <= last ? (int)(last - first + 1u) : 0;
  const int win_first = first <= last ? (int)(first - first_raw_pos) : 0;
  const int wt = (n_win + kTile - 1) / kTile;
  // this workgroup's tiles: all of them, or its share of what the token has at most
  int t_begin = 0, t_share = 0x7FFFFFFF;
  if (CUT && split) {
    t_share = mspr_div(wt + (n_idx + kTile - 1) / kTile + ranges - 1, ranges, inv_ranges);
    t_begin = range * t_share;
  }
  const uint64_t win_base = reinterpret_cast<uint64_t>(win) + (uint64_t)b * (uint64_t)n_raw * (kD * 2);

  // Copies of a tile: this wave's eight rows. `row` holds, per lane l < 32, the row of slot l (-1: no row, zeros).
  const uint32_t lane_off = (uint32_t)lane * 16u;
  const uint32_t my_rows_lds =
      __builtin_amdgcn_readfirstlane((uint32_t)(size_t)MSPR_LDS_PTR(unsigned char, lds) + (uint32_t)(8 * wave * kPitch));
  auto copy_rows = [&](int tile, uint64_t base, int row) {
    const uint32_t dst = my_rows_lds + (uint32_t)((tile & 1) * kTileBytes);
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const int r = __builtin_amdgcn_readlane(row, 8 * wave + j);
      const uint64_t p = r >= 0 ? base + (uint64_t)(uint32_t)r * (kD * 2) : reinterpret_cast<uint64_t>(&g_prefill_zero_row[0]);
      async_row(p, lane_off, dst + (uint32_t)(j * kPitch));
    }
  };
  auto window_row = [&](int tile) -> int {
    const int ls = tile * kTile + (lane & 31);
    uint32_t r = (uint32_t)raw_start + (uint32_t)win_first + (uint32_t)ls;
    if (r >= n_raw) r -= n_raw;
    return ls < n_win ? (int)r : -1;
  };

  // ---- the first window tile needs no ids: on its way before anything else
  if (t_begin < wt) copy_rows(t_begin, win_base, window_row(t_begin));

  // ---- the first ids of a thread, which go to LDS below
  // In a single round of units, cut into ranges, the queries are requested before the ids are looked at, not behind. That takes a
  // trip to memory off a workgroup's start, and pays where all start at once and none follows (60 tokens behind 28000: 34.9 us, and
  // 34.2 with the requests ahead); with more than a round they crowd out the other workgroup's rows (1536 tokens 166.6 and 169.6),
  // and the choice itself costs whole units 0.5 %.
  constexpr int kEager = 2;
  const bool ahead = CUT && units <= kRound;  // uniform
  const int32_t* src = idx + (int64_t)seq * n_idx;
  int eager[kEager] = {};
  if (ahead && n_idx > 0) {
#pragma unroll
    for (int j = 0; j < kEager; j++) {
      const int i = tid + j * kThreads;
      eager[j] = src[i < n_idx ? i : 0];
    }
  }
  if (tid == 0) *stop_sh = n_idx;
  __syncthreads();

  // ---- ids to LDS, position of the first one that ends the walk
  auto stage_ids = [&](int done) {
    uint32_t visible = a.ratio == 0u ? (uint32_t)a.n_pool : (qpos + 1u) / a.ratio;
    if (visible > (uint32_t)a.n_pool) visible = (uint32_t)a.n_pool;
    int found = n_idx;
    auto look = [&](int i, int id) {
      ids[i] = id;
      if (id >= 0 && (uint32_t)id >= visible && i < found) found = i;
    };
#pragma unroll
    for (int j = 0; j < kEager; j++)
      if (j < done && tid + j * kThreads < n_idx) look(tid + j * kThreads, eager[j]);
    for (int i = tid + done * kThreads; i < n_idx; i += kThreads) look(i, src[i]);
    if (found < n_idx) atomicMin(stop_sh, found);
  };
  if (!ahead) stage_ids(0);

  // ---- query operand: lane (head c16, kg) holds q[head][32 ks + 8 kg .. +7], zero rows past n_heads
  const int head = hb * 64 + 16 * wave + c16;
  const bool live = head < a.n_heads;
  const int64_t qoff = (int64_t)b * a.q_batch_stride + (int64_t)t * a.q_token_stride +
                       (int64_t)(live ? head : 0) * a.q_head_stride + 8 * kg;
  f32x4_t raw[QDT == MSPR_F16 ? 1 : 2 * kQSteps];
  u32x4_t qf[kQSteps];
#pragma unroll
  for (int ks = 0; ks < kQSteps; ks++) {
    if constexpr (QDT == MSPR_F16) {
      qf[ks] = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const uint16_t*>(a.q) + qoff + 32 * ks);
    } else {
      const f32x4_t* p = reinterpret_cast<const f32x4_t*>(reinterpret_cast<const float*>(a.q) + qoff + 32 * ks);
      raw[2 * ks] = p[0];
      raw[2 * ks + 1] = p[1];
    }
  }
  if (ahead) stage_ids(kEager);
#pragma unroll
  for (int ks = 0; ks < kQSteps; ks++) {
    if constexpr (QDT != MSPR_F16) {
      const f32x4_t lo = raw[2 * ks], hi = raw[2 * ks + 1];
      qf[ks] = u32x4_t{pack_h2(lo.x, lo.y), pack_h2(lo.z, lo.w), pack_h2(hi.x, hi.y), pack_h2(hi.z, hi.w)};
    }
    if (!live) qf[ks] = u32x4_t{0u, 0u, 0u, 0u};
  }
  const float sink = live && a.sinks ? a.sinks[head] * 1.4426950408889634f : -__builtin_inff();
  __syncthreads();
  const int stop = __builtin_amdgcn_readfirstlane(*stop_sh);
  int n_tiles = wt + (stop + kTile - 1) / kTile;
  if (CUT && n_tiles - t_begin > t_share) n_tiles = t_begin + t_share;

  auto pool_row = [&](int tile) -> int {
    const int gi = (tile - wt) * kTile + (lane & 31);
    const int id = ids[gi < kMaxIds ? gi : 0];
    return gi < stop ? (id >= 0 ? id : -1) : -1;  // (an id in front of the stop is inside the visible prefix)
  };
  const uint64_t pool_base = reinterpret_cast<uint64_t>(a.pool) + (uint64_t)b * (uint64_t)a.n_pool * (kD * 2);
  // rows and validity word of a tile
  auto rows_of = [&](int tile) -> int { return tile < wt ? window_row(tile) : pool_row(tile); };
  int row = rows_of(t_begin);
  if (t_begin >= wt && t_begin < n_tiles) copy_rows(t_begin, pool_base, row);

  f32x4_t oacc[32];
#pragma unroll
  for (int mt = 0; mt < 32; mt++) oacc[mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m_run = -__builtin_inff();  // reference maximum of head c16 (log2 domain), the same in its four lanes
  float l_run = 0.0f;               // this lane's share of the denominator: its eight keys of every tile
  constexpr float kGrow = 8.0f;     // float16 weights stay below 2^8

  const int a_off = c16 * kPitch + 16 * kg;
  const int tr_off = (4 * kg + (c16 >> 2)) * kPitch + 8 * (c16 & 3);

  for (int tile = t_begin; tile < n_tiles; tile++) {
    const uint32_t valid = (uint32_t)__ballot(row >= 0);  // bit l: slot l (both halves of the wave hold the 32 slots)
    // the copies of this tile have landed (they are the only vector-memory operations in flight), and every wave is done
    // with the tile before it, whose buffer the next copies overwrite
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (tile + 1 < n_tiles) {
      row = rows_of(tile + 1);
      copy_rows(tile + 1, tile + 1 < wt ? win_base : pool_base, row);
    }
    const unsigned char* kt = lds + (tile & 1) * kTileBytes;

    // ---- S^T blocks: keys 16 u + 4 kg + i of head c16. The operand reads run kAheadK matrix instructions in front of their
    //      use (stated to the scheduler, which keeps two in flight otherwise; an LDS read takes as long as eight of them).
    f32x4_t sacc[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int ks = 0; ks < kQSteps; ks++)
#pragma unroll
      for (int u = 0; u < 2; u++)
        sacc[u] = mfma16(*reinterpret_cast<const u32x4_t*>(kt + a_off + u * (16 * kPitch) + ks * 64), qf[ks], sacc[u]);
    __builtin_amdgcn_sched_group_barrier(0x100, kAheadK, 0);
#pragma unroll
    for (int i = 0; i < 2 * kQSteps - kAheadK; i++) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, kAheadK, 0);

    // ---- online softmax in the log2 domain
    float sv[8];
    float tmax = -__builtin_inff();
    {
      const uint32_t v0 = valid >> (4 * kg), v1 = valid >> (16 + 4 * kg);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        sv[i] = (v0 >> i) & 1u ? sacc[0][i] * a.scale_log2 : -__builtin_inff();
        sv[4 + i] = (v1 >> i) & 1u ? sacc[1][i] * a.scale_log2 : -__builtin_inff();
        tmax = fmaxf(tmax, fmaxf(sv[i], sv[4 + i]));
      }
    }
    tmax = half_wave_max(row_pair_max(tmax));
    const bool grow = tmax > m_run + kGrow;
    if (__any(grow)) {
      const float m_new = grow ? tmax : m_run;
      const float alpha = grow ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.0f;
      l_run *= alpha;
      m_run = m_new;
#pragma unroll
      for (int mt = 0; mt < 32; mt++) oacc[mt] = oacc[mt] * alpha;
    }
    const float m_safe = m_run == -__builtin_inff() ? 0.0f : m_run;
    u32x4_t pf;
    {
      float p[8];
#pragma unroll
      for (int i = 0; i < 8; i++) {
        p[i] = __builtin_amdgcn_exp2f(sv[i] - m_safe);
        l_run += p[i];
      }
      pf = u32x4_t{pack_h2(p[0], p[1]), pack_h2(p[2], p[3]), pack_h2(p[4], p[5]), pack_h2(p[6], p[7])};
    }

    // ---- O^T += V^T.P^T: output columns 16 mt + 4 kg + i of head c16
#pragma unroll
    for (int mt = 0; mt < 32; mt++) {
      const unsigned char* base = kt + tr_off + mt * 32;
      const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(MSPR_LDS_PTR(s16x4_t, base));
      const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(MSPR_LDS_PTR(s16x4_t, base + 16 * kPitch));
      const u32x2_t lo2 = __builtin_bit_cast(u32x2_t, lo), hi2 = __builtin_bit_cast(u32x2_t, hi);
      oacc[mt] = mfma16(u32x4_t{lo2.x, lo2.y, hi2.x, hi2.y}, pf, oacc[mt]);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * kAheadV, 0);
#pragma unroll
    for (int i = 0; i < 32 - kAheadV; i++) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, kAheadV, 0);
  }

  // ---- sink, normalisation, output
  float l = l_run;
  l += __shfl_xor(l, 16, MSPR_WAVE);
  l += __shfl_xor(l, 32, MSPR_WAVE);
  if (CUT && split) {  // unnormalised, as the registers hold it
    const int part = unit * ranges + range;
    float* po = a.parts + (int64_t)part * (64 * kD) + (wave * 32 * 64 + lane) * 4;
#pragma unroll
    for (int mt = 0; mt < 32; mt++) *reinterpret_cast<f32x4_t*>(po + mt * 256) = oacc[mt];
    if (kg == 0) {
      float* ml = a.parts + (int64_t)split_units * ranges * (64 * kD) + ((int64_t)part * 64 + 16 * wave + c16) * 2;
      ml[0] = m_run;
      ml[1] = l;
    }
    return;
  }
  const float m_all = fmaxf(m_run, sink);
  const float m_safe = m_all == -__builtin_inff() ? 0.0f : m_all;
  const float w = __builtin_amdgcn_exp2f(m_run - m_safe);
  l = l * w + __builtin_amdgcn_exp2f(sink - m_safe);
  const float f = l == 0.0f ? 0.0f : w / l;
  // The accumulators hold 64-byte pieces of 16 heads' rows. They change places through LDS (the tile buffers are free), half
  // of the columns at a time, so that every store writes 1 KB of one row; and as nobody reads 128 KB per token back before
  // the chunk is through, past the caches.
  __syncthreads();
  float* stage = reinterpret_cast<float*>(lds) + wave * (16 * kOutPitch);  // [16 heads][kOutPitch], this wave's own
  float* out = a.out + (int64_t)b * a.q_batch_stride + (int64_t)t * a.q_token_stride +
               (int64_t)(hb * 64 + 16 * wave) * a.q_head_stride + 4 * lane;
  const int n_live = a.n_heads - (hb * 64 + 16 * wave);
#pragma unroll
  for (int half = 0; half < 2; half++) {
#pragma unroll
    for (int mt = 0; mt < 16; mt++)
      *reinterpret_cast<f32x4_t*>(stage + c16 * kOutPitch + 16 * mt + 4 * kg) = oacc[16 * half + mt] * f;
    f32x4_t r[16];
#pragma unroll
    for (int h = 0; h < 16; h++) r[h] = *reinterpret_cast<const f32x4_t*>(stage + h * kOutPitch + 4 * lane);
    if (n_live >= 16) {
#pragma unroll
      for (int h = 0; h < 16; h++)
        __builtin_nontemporal_store(r[h], reinterpret_cast<f32x4_t*>(out + h * a.q_head_stride + 256 * half));
    } else {
#pragma unroll
      for (int h = 0; h < 16; h++)
        if (h < n_live) *reinterpret_cast<f32x4_t*>(out + h * a.q_head_stride + 256 * half) = r[h];
    }
  }
}

// The ranges of the cut units and the sink, normalised. A wave takes one accumulator register quad (16 heads, 16 columns) of
// a unit: every range's is 1 KB, and all are requested at once.
__global__ __launch_bounds__(256) void indexed_prefill_merge_kernel(const float* parts, const float* sinks, int split_units,
                                                                    int ranges, int n_heads, int n_hblk, uint32_t inv_hblk,
                                                                    int n_tokens, uint32_t inv_tokens, float* out,
                                                                    int64_t batch_stride, int64_t token_stride,
                                                                    int64_t head_stride) {
  const int lane = threadIdx.x & 63;
  const int c16 = lane & 15, kg = lane >> 4;
  const int piece = __builtin_amdgcn_readfirstlane((int)blockIdx.x * 4 + (int)(threadIdx.x >> 6));
  const int unit = piece >> 7, wave = (piece >> 5) & 3, mt = piece & 31;
  const int seq = mspr_div(unit, n_hblk, inv_hblk), hb = unit - seq * n_hblk;
  const int b = mspr_div(seq, n_tokens, inv_tokens), t = seq - b * n_tokens;
  const int head = hb * 64 + 16 * wave + c16;
  const float* po = parts + (int64_t)unit * ranges * (64 * kD) + ((wave * 32 + mt) * 64 + lane) * 4;
  const float* ml = parts + (int64_t)split_units * ranges * (64 * kD) + ((int64_t)unit * ranges * 64 + 16 * wave + c16) * 2;
  float m[kMaxRanges], l[kMaxRanges];
  f32x4_t o[kMaxRanges];
#pragma unroll
  for (int r = 0; r < kMaxRanges; r++) {
    const int rr = r < ranges ? r : 0;
    m[r] = ml[rr * 128];
    l[r] = ml[rr * 128 + 1];
    o[r] = *reinterpret_cast<const f32x4_t*>(po + (int64_t)rr * (64 * kD));
    if (r >= ranges) m[r] = -__builtin_inff();
  }
  const float sink = head < n_heads && sinks ? sinks[head] * 1.4426950408889634f : -__builtin_inff();
  float m_all = sink;
#pragma unroll
  for (int r = 0; r < kMaxRanges; r++) m_all = fmaxf(m_all, m[r]);
  const float m_safe = m_all == -__builtin_inff() ? 0.0f : m_all;
  float den = __builtin_amdgcn_exp2f(sink - m_safe);
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int r = 0; r < kMaxRanges; r++) {
    const float w = __builtin_amdgcn_exp2f(m[r] - m_safe);
    den += l[r] * w;
    acc += o[r] * w;
  }
  const float f = den == 0.0f ? 0.0f : 1.0f / den;
  if (head < n_heads)
    *reinterpret_cast<f32x4_t*>(out + (int64_t)b * batch_stride + (int64_t)t * token_stride + (int64_t)head * head_stride +
                                16 * mt + 4 * kg) = acc * f;
}

template <int QDT, bool CUT>
int launch(const IndexedPrefillArgs& a, hipStream_t st) {
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&indexed_prefill_kernel<QDT, CUT>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
    if (e != hipSuccess) {
      mspr_set_error("indexed prefill attention: cannot reserve %d bytes of LDS: %s", kLdsBytes, hipGetErrorString(e));
      return MSPR_ERR_LAUNCH;
    }
    attr_set = true;
  }
  const int n_hblk = (a.n_heads + 63) / 64;
  const int64_t units = (int64_t)a.batch * a.n_tokens * n_hblk;
  dim3 grid((unsigned)(units - a.split_units + a.split_units * a.ranges)), block(kThreads);
  {
    MsprProfScope prof(MSPR_K_SPARSE_SPLIT, st);
    indexed_prefill_kernel<QDT, CUT><<<grid, block, kLdsBytes, st>>>(
        a.win, a.idx, (int)units, a.n_tokens, n_hblk, a.pos0, a.window, (uint32_t)a.raw_cap, a.raw_start, a.n_idx,
        (uint32_t)a.split_units | (uint32_t)a.ranges << 16, mspr_inverse(a.ranges), a);
  }
  MSPR_CHECK_LAUNCH("indexed prefill attention");
  if constexpr (CUT) {
    MsprProfScope prof(MSPR_K_SPARSE_MERGE, st);
    indexed_prefill_merge_kernel<<<dim3((unsigned)(a.split_units * 32)), block, 0, st>>>(
        a.parts, a.sinks, a.split_units, a.ranges, a.n_heads, n_hblk, mspr_inverse(n_hblk), a.n_tokens, mspr_inverse(a.n_tokens), a.out,
        a.q_batch_stride, a.q_token_stride, a.q_head_stride);
    MSPR_CHECK_LAUNCH("indexed prefill attention (merge)");
  }
  return MSPR_OK;
}

}  // namespace

bool mspr_indexed_prefill_fits(int batch, int n_heads, int n_tokens, int n_idx) {
  return n_idx <= kMaxIds && (int64_t)batch * n_tokens * ((n_heads + 63) / 64) < ((int64_t)1 << 31);
}

static int tiles_of(int64_t rows) { return (int)((rows + kTile - 1) / kTile); }

// Two workgroups on each of 256 CUs are a round; what is left of the last one runs one to a CU, and if it is few units the
// chip is idle. They are cut into as many key ranges as keep the partials (128 KB each) under 24 MB, or, where those would
// be one or two and no round is in front, as leave one workgroup to a CU; with at least two id tiles in each. Whether that
// pays is estimated: a tile takes 1.13 us alone and about 1 us under the round in front, and the partials and their merge
// cost what was fitted to 1 to 96 units of 128 to 1024 ids and a window of 128, whole and in 2 to 8 ranges (float16 and
// float32 queries, pools of 1200 to 6000 rows). Whole and cut, us: 512 ids 1 token 30 and 13, 16 tokens 31 and 21, 64
// tokens 31 and 27, 80 tokens 31 and 29 (in two ranges 32), 96 tokens 31 and 34 (left whole); 513 tokens 73 and 58, 576
// tokens 75 and 71. 256 ids 24 tokens 21.5 and 19.9, 48 tokens 21.5 and 23.2 (left whole). 128 ids 8 tokens 16.6 and 14.9,
// 24 tokens 16.9 and 18.0, 64 tokens 17 and 25 (left whole), 520 tokens 40.7 and 40.2, 560 tokens 41.2 and 44.4 (left
// whole).
// The kernel deals out the tiles of a window of `window_rows` and all of a token's ids; `tiles` of them hold rows at most.
static void cut_last_round(IndexedPrefillArgs& a, int64_t window_rows, int tiles) {
  const int64_t units = (int64_t)a.batch * a.n_tokens * ((a.n_heads + 63) / 64);
  const int left = (int)(units % 512);
  const bool alone = units < 512;
  int ranges = left == 0 ? 1 : (alone && left > 64 ? 256 : 192) / left;
  if (ranges > a.n_idx / (2 * kTile)) ranges = a.n_idx / (2 * kTile);
  if (ranges > kMaxRanges) ranges = kMaxRanges;
  a.split_units = 0;
  a.ranges = 1;
  if (ranges < 2) return;
  const float tile_us = alone ? 1.13f : 1.0f, parts = (float)(left * ranges);
  // (many partials of long ranges, which are all written at once, cost 2 us more)
  const float merge_us = alone ? 2.5f + (parts < 110.0f ? 0.065f * parts : 7.15f + 0.02f * (parts - 110.0f) +
                                                                              (ranges == 2 ? 2.0f : 0.0f))
                               : 3.0f + 0.035f * parts;
  const int share = (tiles_of(window_rows) + tiles_of(a.n_idx) + ranges - 1) / ranges;
  if (tile_us * (float)(share < tiles ? share : tiles) + merge_us >= tile_us * (float)tiles - 0.3f) return;
  a.split_units = left;
  a.ranges = ranges;
}

static size_t part_bytes(const IndexedPrefillArgs& a) {
  return (size_t)a.split_units * a.ranges * (64 * kD + 64 * 2) * sizeof(float);
}

size_t mspr_indexed_prefill_workspace_bytes(int batch, int n_heads, int n_tokens, int window_rows, int n_idx) {
  IndexedPrefillArgs a = {};
  a.batch = batch;
  a.n_heads = n_heads;
  a.n_tokens = n_tokens;
  a.n_idx = n_idx;
  cut_last_round(a, window_rows, tiles_of(window_rows) + tiles_of(n_idx));
  return part_bytes(a);
}

int mspr_launch_indexed_prefill(const IndexedPrefillArgs& call, void* workspace, size_t workspace_bytes, hipStream_t st) {
  IndexedPrefillArgs a = call;
  // The units that may be cut are the first tokens' (of the first sequence): the rows that those see at most. (The workspace
  // was sized without their position, for all rows; where it is too small for the ranges chosen here, there are fewer.)
  const int64_t units = (int64_t)a.batch * a.n_tokens * ((a.n_heads + 63) / 64);
  const int64_t last = units % 512 / ((a.n_heads + 63) / 64);
  const int64_t seen = (int64_t)a.pos0 + (last < a.n_tokens ? last : a.n_tokens);
  int64_t ids = a.ratio == 0u ? a.n_pool : seen / a.ratio;
  if (ids > a.n_pool) ids = a.n_pool;
  if (ids > a.n_idx) ids = a.n_idx;
  cut_last_round(a, a.max_win, tiles_of(a.max_win < seen ? a.max_win : seen) + tiles_of(ids));
  a.parts = static_cast<float*>(workspace);
  if (!workspace || !mspr_aligned(workspace, 16)) a.split_units = 0;
  while (a.ranges > 1 && workspace_bytes < part_bytes(a)) a.ranges--;
  if (a.ranges == 1) a.split_units = 0;
  if (a.split_units == 0) a.ranges = 1;
  if (a.split_units > 0) return a.q_dtype == MSPR_F32 ? launch<MSPR_F32, true>(a, st) : launch<MSPR_F16, true>(a, st);
  return a.q_dtype == MSPR_F32 ? launch<MSPR_F32, false>(a, st) : launch<MSPR_F16, false>(a, st);
}
