// Deterministic top-k over float32 score rows: select on monotone uint32 keys, then ordered emission
// (rows strictly above the k-th key in ascending row order, then the lowest-index rows tied with it).
//
// One workgroup per score row; which kernel depends on the row's length, k and the number of rows (mspr_launch_topk):
//  * topk_sampled_kernel, rows of 2049 to 32768 scores of which a small part is wanted: the keys above a sampled pivot are
//    listed, binned and ranked.
//  * topk_row_kernel, rows of up to 8192: the keys stay in registers and are binned by value range.
//  * topk_blocked_kernel, the others of up to 32768: a thread owns consecutive rows; a list above a pivot up to 8192 scores,
//    else four 8-bit digits from the top over all keys.
//  * topk_select_kernel, longer rows: the same digits, global memory re-read each pass.
// Samples and pivots decide how long a call takes, never what it returns: that a list holds the k-th key is checked exactly.
//
// Digit histograms over all keys are 256 bins x 64 copies in LDS, copy = lane id, laid out [bin][copy], so every lane of an
// LDS atomic hits its own bank whatever the digit distribution is (scores of one row usually share their top byte, which
// would serialise a single shared counter 64-fold). After two digits the keys that still match the prefix are usually a
// handful; they are compacted into an LDS list and the last two digits run on that list only.
#include <cmath>

#include "common.h"
#include "profile.h"

namespace {

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / 64;
constexpr int kCopies = 64;
constexpr int kListCap = 2048;
constexpr int kFastPer = 6;                     // survivor-list entries per thread on the pivot path
constexpr int kFastCap = kFastPer * kThreads;   // survivor-list capacity

struct SelectState {
  uint32_t prefix;
  uint32_t need;
  uint32_t live;   // keys matching the current prefix
  uint32_t list_n;
};

// Wave 0: pick the bucket where the count from the top first reaches `need`. totals[b] in LDS.
__device__ __forceinline__ void choose_bucket(const uint32_t* totals, SelectState* st, uint32_t shift, int lane) {
  uint32_t t[4];
#pragma unroll
  for (int j = 0; j < 4; j++) t[j] = totals[4 * lane + j];
  uint32_t lane_sum = t[0] + t[1] + t[2] + t[3];
  uint32_t sfx = lane_sum;  // inclusive suffix sum over lanes
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    uint32_t o = __shfl_down(sfx, off, MSPR_WAVE);
    if (lane + off < 64) sfx += o;
  }
  const uint32_t need = st->need;
  const uint32_t prefix = st->prefix;
  int chosen = -1;
  uint32_t chosen_need = 0u, chosen_cnt = 0u;
  uint32_t run = sfx - lane_sum;  // keys in buckets of higher lanes
#pragma unroll
  for (int j = 3; j >= 0; j--) {
    if (chosen < 0 && run < need && run + t[j] >= need) {
      chosen = 4 * lane + j;
      chosen_need = need - run;
      chosen_cnt = t[j];
    }
    run += t[j];
  }
  uint64_t any = __ballot(chosen >= 0);
  if (any == 0ull) {
    // fewer live keys than needed cannot happen for topk <= n_rows; bucket 0 takes the rest
    if (lane == 0) {
      st->need = need - (sfx - t[0]);
      st->live = t[0];
    }
  } else if (chosen >= 0) {
    st->prefix = prefix | ((uint32_t)chosen << shift);
    st->need = chosen_need;
    st->live = chosen_cnt;
  }
}

__global__ __launch_bounds__(kThreads) void topk_select_kernel(const float* __restrict__ scores_all,
                                                                int64_t score_stride, int64_t n_rows, int topk,
                                                                int32_t* __restrict__ sel_all) {
  __shared__ uint32_t hist[256 * kCopies];  // [bin][copy]
  __shared__ uint32_t totals[256];
  __shared__ uint32_t list[kListCap];
  __shared__ SelectState st;
  __shared__ uint32_t cnt_above[kThreads];
  __shared__ uint32_t cnt_tie[kThreads];
  __shared__ uint32_t wave_tot[2 * kWaves];
  __shared__ uint32_t carry[2];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const float* scores = scores_all + (int64_t)blockIdx.x * score_stride;
  int32_t* sel = sel_all + (int64_t)blockIdx.x * topk;
  const int64_t n_chunks = (n_rows + kThreads - 1) / kThreads;

  if (tid == 0) {
    st.prefix = 0u;
    st.need = (uint32_t)topk;
    st.live = (uint32_t)n_rows;
    st.list_n = 0u;
  }

  // one digit over every key: count keys whose higher digits equal the prefix
  auto full_pass = [&](int pass) {
    const uint32_t shift = 24u - 8u * pass;
    u32x4_t* h4 = reinterpret_cast<u32x4_t*>(hist);
    for (int i = tid; i < 256 * kCopies / 4; i += kThreads) h4[i] = u32x4_t{0u, 0u, 0u, 0u};
    __syncthreads();
    const uint32_t prefix = st.prefix;
    const uint32_t mask_hi = pass == 0 ? 0u : (0xFFFFFFFFu << (shift + 8u));
    for (int64_t c = 0; c < n_chunks; c++) {
      int64_t r = c * kThreads + tid;
      if (r < n_rows) {
        uint32_t key = score_key(scores[r]);
        if ((key & mask_hi) == prefix) atomicAdd(&hist[((key >> shift) & 0xFFu) * kCopies + lane], 1u);
      }
    }
    __syncthreads();
    // totals[bin] = sum over copies: four threads per bin, 16 copies each, rotated to spread banks
    {
      const int bin = tid >> 2, q = tid & 3;
      uint32_t s = 0u;
#pragma unroll
      for (int j = 0; j < 16; j++) s += hist[bin * kCopies + q * 16 + ((j + lane) & 15)];
      s += __shfl_xor(s, 1, MSPR_WAVE);
      s += __shfl_xor(s, 2, MSPR_WAVE);
      if (q == 0) totals[bin] = s;
    }
    __syncthreads();
    if (wave == 0) choose_bucket(totals, &st, shift, lane);
    __syncthreads();
  };

  full_pass(0);
  full_pass(1);

  if (st.live <= (uint32_t)kListCap) {
    // compact the keys that match the 16-bit prefix; their order does not matter here
    const uint32_t prefix = st.prefix;
    for (int64_t c = 0; c < n_chunks; c++) {
      int64_t r = c * kThreads + tid;
      if (r < n_rows) {
        uint32_t key = score_key(scores[r]);
        if ((key & 0xFFFF0000u) == prefix) list[atomicAdd(&st.list_n, 1u)] = key;
      }
    }
    __syncthreads();
    const uint32_t n_list = st.list_n;
    for (int pass = 2; pass < 4; pass++) {
      const uint32_t shift = 24u - 8u * pass;
      if (tid < 256) totals[tid] = 0u;
      __syncthreads();
      const uint32_t pfx = st.prefix;
      const uint32_t mask_hi = 0xFFFFFFFFu << (shift + 8u);
      for (uint32_t i = tid; i < n_list; i += kThreads) {
        uint32_t key = list[i];
        if ((key & mask_hi) == pfx) atomicAdd(&totals[(key >> shift) & 0xFFu], 1u);
      }
      __syncthreads();
      if (wave == 0) choose_bucket(totals, &st, shift, lane);
      __syncthreads();
    }
  } else {
    full_pass(2);
    full_pass(3);
  }

  const uint32_t threshold = st.prefix;
  const uint32_t need_ties = st.need;
  const uint32_t n_above = (uint32_t)topk - need_ties;
  if (tid == 0) {
    carry[0] = 0u;
    carry[1] = 0u;
  }
  __syncthreads();

  // Emission in groups of 64 chunks (65536 rows): per (chunk, wave) counts -> one block scan.
  const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  auto count_chunk = [&](int ci, bool live, uint32_t key) {
    uint64_t ba = __ballot(live && key > threshold);
    uint64_t bt = __ballot(live && key == threshold);
    if (lane == 0) {
      cnt_above[ci * kWaves + wave] = (uint32_t)__popcll(ba);
      cnt_tie[ci * kWaves + wave] = (uint32_t)__popcll(bt);
    }
  };
  auto emit_chunk = [&](int ci, int64_t r, bool live, uint32_t key) {
    bool is_above = live && key > threshold;
    bool is_tie = live && key == threshold;
    uint64_t ba = __ballot(is_above);
    uint64_t bt = __ballot(is_tie);
    if (is_above) {
      uint32_t slot = cnt_above[ci * kWaves + wave] + (uint32_t)__popcll(ba & lt_mask);
      sel[slot] = (int32_t)r;
    } else if (is_tie) {
      uint32_t rank = cnt_tie[ci * kWaves + wave] + (uint32_t)__popcll(bt & lt_mask);
      if (rank < need_ties) sel[n_above + rank] = (int32_t)r;
    }
  };
  for (int64_t g0 = 0; g0 < n_chunks; g0 += 64) {
    const int gchunks = (int)((n_chunks - g0) < 64 ? (n_chunks - g0) : 64);
    for (int ci = 0; ci < gchunks; ci++) {
      int64_t r = (g0 + ci) * kThreads + tid;
      bool live = r < n_rows;
      count_chunk(ci, live, live ? score_key(scores[r]) : 0u);
    }
    for (int i = gchunks * kWaves + tid; i < kThreads; i += kThreads) {
      cnt_above[i] = 0u;
      cnt_tie[i] = 0u;
    }
    __syncthreads();
    // exclusive scan over the (chunk, wave) entries, one per thread
    uint32_t va = cnt_above[tid], vt = cnt_tie[tid];
    uint32_t ia = va, it = vt;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      uint32_t oa = __shfl_up(ia, off, MSPR_WAVE);
      uint32_t ot = __shfl_up(it, off, MSPR_WAVE);
      if (lane >= off) {
        ia += oa;
        it += ot;
      }
    }
    if (lane == 63) {
      wave_tot[wave] = ia;
      wave_tot[kWaves + wave] = it;
    }
    __syncthreads();
    uint32_t base_a = carry[0], base_t = carry[1];
    for (int w = 0; w < wave; w++) {
      base_a += wave_tot[w];
      base_t += wave_tot[kWaves + w];
    }
    __syncthreads();
    cnt_above[tid] = base_a + ia - va;
    cnt_tie[tid] = base_t + it - vt;
    if (tid == kThreads - 1) {
      carry[0] = base_a + ia;
      carry[1] = base_t + it;
    }
    __syncthreads();
    for (int ci = 0; ci < gchunks; ci++) {
      int64_t r = (g0 + ci) * kThreads + tid;
      bool live = r < n_rows;
      emit_chunk(ci, r, live, live ? score_key(scores[r]) : 0u);
    }
    __syncthreads();
  }
}

// Every wave runs this on the same 256 totals and gets the same answer in every lane: the digit
// where the count from the top first reaches `need`, the keys still needed inside it and its size.
struct Pick {
  uint32_t digit, need, live;
};
// Inclusive prefix sum over the 64 lanes with data-parallel-primitive moves (no LDS round trips):
// four shifts inside each row of 16 lanes, then the row totals are carried across rows.
__device__ __forceinline__ uint32_t wave_prefix_sum(uint32_t x) {
  int v = (int)x;
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // row_bcast:15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // row_bcast:31 into rows 2 and 3
  return (uint32_t)v;
}

// mask = 2 mask + bit
__device__ __forceinline__ uint32_t shift_in(uint32_t mask, bool bit) { return (mask << 1) | (bit ? 1u : 0u); }

// One histogram vote per lane. Up to four rounds first count all lanes that share the bin of the
// lowest voting lane with a single atomic (digits near the top of the key are shared by most rows,
// which would serialise one atomic per lane on the same counter); what is left votes directly.
__device__ __forceinline__ void wave_hist_add(uint32_t* h, int bin, int lane) {
#pragma unroll
  for (int round = 0; round < 4; round++) {
    const uint64_t voters = __ballot(bin >= 0);
    if (voters == 0ull) break;
    const int first = (int)__builtin_ctzll(voters);
    const int d = __builtin_amdgcn_readlane(bin, first);
    const uint64_t same = __ballot(bin == d);
    if (lane == first) atomicAdd(&h[d], (uint32_t)__popcll(same));
    if (bin == d) bin = -1;
  }
  if (bin >= 0) atomicAdd(&h[bin], 1u);
}

__device__ __forceinline__ Pick pick_bucket(const uint32_t* totals, uint32_t need, int lane) {
  // lane l looks at digits 255-4l .. 252-4l, so a prefix sum over lanes counts keys from the top digit down
  uint32_t t[4];
#pragma unroll
  for (int j = 0; j < 4; j++) t[j] = totals[255 - (4 * lane + j)];
  const uint32_t lane_sum = t[0] + t[1] + t[2] + t[3];
  const uint32_t incl = wave_prefix_sum(lane_sum);
  int chosen = -1;
  uint32_t chosen_need = 0u, chosen_cnt = 0u;
  uint32_t run = incl - lane_sum;  // keys in higher digits
#pragma unroll
  for (int j = 0; j < 4; j++) {
    if (chosen < 0 && run < need && run + t[j] >= need) {
      chosen = 255 - (4 * lane + j);
      chosen_need = need - run;
      chosen_cnt = t[j];
    }
    run += t[j];
  }
  const uint64_t any = __ballot(chosen >= 0);
  Pick p;
  if (any) {
    const int src = (int)__builtin_ctzll(any);
    p.digit = (uint32_t)__builtin_amdgcn_readlane(chosen, src);
    p.need = (uint32_t)__builtin_amdgcn_readlane((int)chosen_need, src);
    p.live = (uint32_t)__builtin_amdgcn_readlane((int)chosen_cnt, src);
  } else {
    // fewer keys than needed cannot happen for topk <= rows held; digit 0 would take the rest
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    const uint32_t d0 = (uint32_t)__builtin_amdgcn_readlane((int)t[3], 63);
    p.digit = 0u;
    p.need = need - (total - d0);
    p.live = d0;
  }
  return p;
}

// Rows of up to C*1024 scores: thread t owns the C consecutive rows [C t, C t + C) in registers.
// With consecutive ownership the ordered emission needs no cross-lane work per row: a thread knows
// the relative order of its own rows, so one packed block scan of the per-thread counts gives every
// thread its output slots. Digit histograms over all keys use 256 bins x 64 copies (copy = lane, so
// an LDS atomic never meets a bank conflict whatever the digit distribution); the thread that sums a
// group of copies also zeroes it for the next pass. Select state lives in registers: every wave derives it
// from the same totals, which saves the broadcast barriers.
// Rows past n_rows are given key 0: they can only tie with the lowest possible key and lose every
// tie to a real row (ties go to the lower index), so no pass needs a bounds check.
// (The sampled kernel further down takes the rows of which a small part is wanted; the pivot path here is for those of up to
// 8192 scores with more. Of longer rows, none that is left has a pivot whose keys would fit the list.)
static_assert(kFastCap / 2 >= kListCap, "the list of the full passes fits the space of the pivot path's");
template <int C, bool PIVOT>
__global__ __launch_bounds__(kThreads) void topk_blocked_kernel(const float* __restrict__ scores_all,
                                                                 int64_t score_stride, int n_rows, int topk,
                                                                 int sample_rank, int32_t* __restrict__ sel_all) {
  // The staging area for the load (C*1024 keys) is reused for the histogram copies afterwards.
  // copies of the full-pass histograms: one per lane where the staging area is that large anyway; 32 (lanes l and
  // l + 32 share one) for the short-row instance, whose LDS then lets two workgroups share a CU
  constexpr int kCp = C * kThreads >= 256 * kCopies ? kCopies : kCopies / 2;
  constexpr int kStageWords = C * kThreads > 256 * kCp ? C * kThreads : 256 * kCp;
  __shared__ __attribute__((aligned(16))) uint32_t stage[kStageWords];
  uint32_t* hist = stage;                   // [bin][copy]
  __shared__ uint32_t totals[256];
  __shared__ uint32_t small_hist[2][256];   // digits 2 and 3 on the compacted list
  // survivor rows of the pivot path (16-bit row numbers), or the compacted keys of the full passes
  __shared__ __attribute__((aligned(16))) uint32_t list_words[PIVOT ? kFastCap / 2 : kListCap];
  uint32_t* list = list_words;
  uint16_t* fast_rows = reinterpret_cast<uint16_t*>(list_words);
  __shared__ uint32_t list_n;
  __shared__ uint32_t wave_tot[kWaves];
  __shared__ uint32_t fhist[5][256];        // pivot path: two sample digits, three digits on the survivor list
  __shared__ Pick pick_box[5];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const float* scores = scores_all + (int64_t)blockIdx.x * score_stride;
  int32_t* sel = sel_all + (int64_t)blockIdx.x * topk;
  if (PIVOT && sample_rank > 0)
    for (int i = tid; i < 5 * 256; i += kThreads) (&fhist[0][0])[i] = 0u;  // ordered by the barriers of the load

  // Load with lane-contiguous 16-byte reads (a wave reads 1 KB at a time), then hand every thread its
  // C consecutive rows through LDS. The 16-byte pieces of a thread's C/4-piece block are XOR-permuted
  // by the thread index so that neither the writes nor the reads pile up on a few banks.
  uint32_t kreg[C];
  constexpr int kPieces = C / 4;  // 16-byte pieces per thread
  {
    // (rows of a batch start at any multiple of 4 bytes; the 16-byte loads need no more than that. Element by element a row
    // that starts off 16 bytes took 5 us longer: 5 rows of 19211 scores, k = 1024: 13.6 -> 10.7 us)
    typedef __attribute__((ext_vector_type(4), aligned(4))) float f32x4_any_t;
    const bool vec_ok = n_rows >= 4;  // uniform
    // all vector loads first, unconditionally (a piece that crosses the end of the row re-reads the
    // last whole piece and is patched element by element below)
    f32x4_t v[kPieces];
    const int last_whole = (n_rows - 4) & ~3;
    if (vec_ok) {
#pragma unroll
      for (int k = 0; k < kPieces; k++) {
        const int r = 4 * (k * kThreads + tid);
        v[k] = *reinterpret_cast<const f32x4_any_t*>(scores + (r < last_whole ? r : last_whole));
      }
    }
#pragma unroll
    for (int k = 0; k < kPieces; k++) {
      const int piece = k * kThreads + tid;  // global piece index: rows 4*piece .. 4*piece+3
      const int r = 4 * piece;
      u32x4_t keys;
      if (vec_ok && r + 3 < n_rows) {
        keys = u32x4_t{score_key(v[k].x), score_key(v[k].y), score_key(v[k].z), score_key(v[k].w)};
      } else if (r < n_rows) {
        float t[4];  // (requested together)
#pragma unroll
        for (int e = 0; e < 4; e++) t[e] = scores[r + e < n_rows ? r + e : n_rows - 1];
#pragma unroll
        for (int e = 0; e < 4; e++) keys[e] = r + e < n_rows ? score_key(t[e]) : 0u;
      } else {
        keys = u32x4_t{0u, 0u, 0u, 0u};
      }
      const int owner = piece / kPieces, j = piece % kPieces;
      *reinterpret_cast<u32x4_t*>(&stage[owner * C + 4 * (j ^ (owner & (kPieces - 1)))]) = keys;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPieces; j++) {
      const u32x4_t keys = *reinterpret_cast<const u32x4_t*>(&stage[tid * C + 4 * (j ^ (tid & (kPieces - 1)))]);
#pragma unroll
      for (int e = 0; e < 4; e++) kreg[4 * j + e] = keys[e];
    }
  }

  // ---- pivot path. Every thread's first row is a sample of the (padded) row set; the 16-bit key
  // prefix at rank `sample_rank` of the sample sits, with a wide margin, below the k-th key of the
  // whole row, so the rows at or above it ("survivors", a few thousand) contain the answer. They are
  // compacted in row order and the exact select and the emission run on that list only. Whether the
  // pivot was good is checked exactly (survivors >= k, within the list capacity, k-th key less than
  // 255 prefixes above the pivot); if not, the full radix passes below take over, so the result never
  // depends on the sample. The keys stay in the staging area, which this path does not overwrite.
  // one wave works out the digit, the others wait for it: with 16 waves on 4 SIMDs a computation that
  // every wave repeats costs four times its instruction count, a barrier costs less (a slot per use,
  // so no slot is rewritten while a slow wave may still read it)
  auto shared_pick = [&](const uint32_t* h, uint32_t want, int slot) -> Pick {
    if (wave == 0) {
      const Pick p = pick_bucket(h, want, lane);
      if (lane == 0) pick_box[slot] = p;
    }
    __syncthreads();
    return pick_box[slot];
  };
  if (PIVOT && sample_rank > 0) {
    const uint32_t skey = kreg[0];
    wave_hist_add(fhist[0], (int)(skey >> 24), lane);  // the top byte is shared by most rows: vote per wave
    __syncthreads();
    const Pick s0 = shared_pick(fhist[0], (uint32_t)sample_rank, 0);
    if ((skey >> 24) == s0.digit) atomicAdd(&fhist[1][(skey >> 16) & 0xFFu], 1u);
    __syncthreads();
    const Pick s1 = shared_pick(fhist[1], s0.need, 1);
    const uint32_t pivot16 = (s0.digit << 8) | s1.digit;
    const uint32_t pivot = pivot16 << 16;

    uint32_t smask = 0u;
#pragma unroll
    for (int i = C - 1; i >= 0; i--) smask = shift_in(smask, kreg[i] >= pivot);
    const uint32_t cnt = (uint32_t)__popc(smask);
    const uint32_t sincl = wave_prefix_sum(cnt);
    if (lane == 63) wave_tot[wave] = sincl;
    __syncthreads();
    uint32_t sbase = 0u, total = 0u;
#pragma unroll
    for (int w = 0; w < kWaves; w++) {
      const uint32_t wt = wave_tot[w];
      sbase += w < wave ? wt : 0u;
      total += wt;
    }
    if (total >= (uint32_t)topk && total <= (uint32_t)kFastCap) {  // the same for every thread
      uint32_t pos = sbase + sincl - cnt;
      while (smask) {
        const int i = __builtin_ctz(smask);
        smask &= smask - 1u;
        fast_rows[pos++] = (uint16_t)(C * tid + i);
      }
      __syncthreads();
      // thread t takes the list entries [t E, t E + E): consecutive, so the emission order is again a
      // matter of one block scan
      const uint32_t per = (total + kThreads - 1) / kThreads;  // 1 .. kFastPer
      uint32_t lk[kFastPer], lr[kFastPer];
      uint32_t lvalid = 0u;
#pragma unroll
      for (int j = 0; j < kFastPer; j++) {
        const uint32_t idx = (uint32_t)tid * per + j;
        const bool ok = (uint32_t)j < per && idx < total;
        const uint32_t row = fast_rows[ok ? idx : 0u];
        const uint32_t owner = row / C, piece = (row % C) >> 2, e = row & 3u;
        lr[j] = row;
        lk[j] = stage[owner * C + 4 * (piece ^ (owner & (kPieces - 1))) + e];
        lvalid |= (ok ? 1u : 0u) << j;
      }
      // digit A: distance of the 16-bit prefix from the pivot's, everything 255 or more prefixes up in
      // one bin; digits B and C: the low 16 bits
      uint32_t* hA = fhist[2];
#pragma unroll
      for (int j = 0; j < kFastPer; j++) {
        const uint32_t d = (lk[j] >> 16) - pivot16;
        if ((lvalid >> j) & 1u) atomicAdd(&hA[d < 255u ? d : 255u], 1u);
      }
      __syncthreads();
      const Pick pa = shared_pick(hA, (uint32_t)topk, 2);
      if (pa.digit < 255u) {  // the same for every thread
        uint32_t fprefix = (pivot16 + pa.digit) << 16, fneed = pa.need;
#pragma unroll
        for (int pass = 2; pass < 4; pass++) {
          const uint32_t shift = 24u - 8u * pass;
          const uint32_t mask_hi = 0xFFFFFFFFu << (shift + 8u);
          uint32_t* h = fhist[1 + pass];
#pragma unroll
          for (int j = 0; j < kFastPer; j++)
            if (((lvalid >> j) & 1u) && (lk[j] & mask_hi) == fprefix) atomicAdd(&h[(lk[j] >> shift) & 0xFFu], 1u);
          __syncthreads();
          const Pick pk = shared_pick(h, fneed, 1 + pass);
          fprefix |= pk.digit << shift;
          fneed = pk.need;
        }
        const uint32_t n_above_f = (uint32_t)topk - fneed;
        uint32_t am = 0u, tm = 0u;
#pragma unroll
        for (int j = 0; j < kFastPer; j++) {
          const bool ok = (lvalid >> j) & 1u;
          am |= (ok && lk[j] > fprefix ? 1u : 0u) << j;
          tm |= (ok && lk[j] == fprefix ? 1u : 0u) << j;
        }
        const uint32_t mine_f = (uint32_t)__popc(am) | ((uint32_t)__popc(tm) << 16);
        const uint32_t incl_f = wave_prefix_sum(mine_f);
        if (lane == 63) wave_tot[wave] = incl_f;  // its earlier contents were consumed before the barriers above
        __syncthreads();
        uint32_t base_f = 0u;
        for (int w = 0; w < wave; w++) base_f += wave_tot[w];
        const uint32_t excl_f = base_f + incl_f - mine_f;
        uint32_t slot_f = excl_f & 0xFFFFu;
        uint32_t rank_f = excl_f >> 16;
#pragma unroll
        for (int j = 0; j < kFastPer; j++) {
          if ((am >> j) & 1u) sel[slot_f++] = (int32_t)lr[j];
          else if (((tm >> j) & 1u) && rank_f < fneed) sel[n_above_f + rank_f++] = (int32_t)lr[j];
        }
        return;
      }
    }
  }
  __syncthreads();  // the staging area and wave_tot have been read by every thread; the full passes reuse them

  {
    u32x4_t* h4 = reinterpret_cast<u32x4_t*>(hist);
    for (int i = tid; i < 256 * kCp / 4; i += kThreads) h4[i] = u32x4_t{0u, 0u, 0u, 0u};
    if (tid < 512) (&small_hist[0][0])[tid] = 0u;
    if (tid == 0) list_n = 0u;
  }
  __syncthreads();

  uint32_t prefix = 0u, need = (uint32_t)topk, live = (uint32_t)(C * kThreads);

  // one digit over every key of the thread
  auto full_pass = [&](int pass) {
    const uint32_t shift = 24u - 8u * pass;
    const uint32_t mask_hi = pass == 0 ? 0u : (0xFFFFFFFFu << (shift + 8u));
#pragma unroll
    for (int i = 0; i < C; i++) {
      const uint32_t key = kreg[i];
      if (pass == 0 || (key & mask_hi) == prefix)
        atomicAdd(&hist[((key >> shift) & 0xFFu) * kCp + (lane & (kCp - 1))], 1u);
    }
    __syncthreads();
    // totals[bin] = sum over copies: four threads per bin, a quarter of the copies each as 16-byte reads
    // (rotated so that 16 neighbouring lanes cover all 16 bank groups), zeroed behind the read
    {
      const int bin = tid >> 2, q = tid & 3;
      uint32_t sum = 0u;
#pragma unroll
      for (int j = 0; j < kCp / 16; j++) {
        u32x4_t* p = reinterpret_cast<u32x4_t*>(&hist[bin * kCp + q * (kCp / 4) + 4 * ((j + (tid >> 2)) & (kCp / 16 - 1))]);
        const u32x4_t v = *p;
        *p = u32x4_t{0u, 0u, 0u, 0u};
        sum += v.x + v.y + v.z + v.w;
      }
      sum += __shfl_xor(sum, 1, MSPR_WAVE);
      sum += __shfl_xor(sum, 2, MSPR_WAVE);
      if (q == 0) totals[bin] = sum;
    }
    __syncthreads();
    const Pick p = pick_bucket(totals, need, lane);
    prefix |= p.digit << shift;
    need = p.need;
    live = p.live;
  };

  full_pass(0);
  full_pass(1);

  if (live <= (uint32_t)kListCap) {
    // the keys that still match the 16-bit prefix are few: finish the select on a compacted list
#pragma unroll
    for (int i = 0; i < C; i++) {
      const uint32_t key = kreg[i];
      if ((key & 0xFFFF0000u) == prefix) list[atomicAdd(&list_n, 1u)] = key;
    }
    __syncthreads();
    const uint32_t n_list = list_n;
#pragma unroll
    for (int pass = 2; pass < 4; pass++) {
      const uint32_t shift = 24u - 8u * pass;
      const uint32_t mask_hi = 0xFFFFFFFFu << (shift + 8u);
      uint32_t* h = small_hist[pass - 2];
      for (uint32_t i = tid; i < n_list; i += kThreads) {
        const uint32_t key = list[i];
        if ((key & mask_hi) == prefix) atomicAdd(&h[(key >> shift) & 0xFFu], 1u);
      }
      __syncthreads();
      const Pick p = pick_bucket(h, need, lane);
      prefix |= p.digit << shift;
      need = p.need;
      live = p.live;
    }
  } else {
    full_pass(2);
    full_pass(3);
  }

  const uint32_t threshold = prefix;
  const uint32_t need_ties = need;
  const uint32_t n_above = (uint32_t)topk - need_ties;

  // ---- ordered emission: per-thread masks, one packed block scan (above count low, tie count high)
  uint32_t above_mask = 0u, tie_mask = 0u;
#pragma unroll
  for (int i = 0; i < C; i++) {
    above_mask |= (kreg[i] > threshold ? 1u : 0u) << i;
    tie_mask |= (kreg[i] == threshold ? 1u : 0u) << i;
  }
  const uint32_t mine = (uint32_t)__popc(above_mask) | ((uint32_t)__popc(tie_mask) << 16);
  const uint32_t incl = wave_prefix_sum(mine);
  if (lane == 63) wave_tot[wave] = incl;
  __syncthreads();
  uint32_t base = 0u;
  for (int w = 0; w < wave; w++) base += wave_tot[w];
  const uint32_t excl = base + incl - mine;
  uint32_t slot_a = excl & 0xFFFFu;
  uint32_t rank_t = excl >> 16;
  const int row0 = C * tid;
  while (above_mask) {
    const int i = __builtin_ctz(above_mask);
    above_mask &= above_mask - 1u;
    sel[slot_a++] = row0 + i;
  }
  while (tie_mask && rank_t < need_ties) {
    const int i = __builtin_ctz(tie_mask);
    tie_mask &= tie_mask - 1u;
    sel[n_above + rank_t++] = row0 + i;
  }
}

// Rows of up to C * THREADS scores, one a workgroup: key j * THREADS + t in register j of thread t. The selection is by
// value range instead of by digit: 1024 bins over the span from a lower bound of the k-th key to the highest key, then the
// bin with the k-th key becomes the span, until it holds 64 keys or fewer, which every wave ranks for itself. The scores
// of a row share their leading bits, so a digit's votes meet on a few counters and take a pass each for four digits;
// the bins of the span spread the votes, and one round is nearly always enough. The lower bound is the lowest of the
// maxima of k or more disjoint groups of keys, or, where a group holds nothing finite, the lowest finite key; -inf (a row
// that a token may not see yet) is then counted on the side and does not stretch the span. Keys past n_rows are 0: they
// can only tie with the lowest possible key and lose every tie to a real row. Emission order comes from ballots: the
// hits of (chunk, wave) pairs are scanned and a wave stores its own side by side.
// What is left is instructions per key and barriers. Four 8-bit digit passes with merged votes took, k = 512: 1 row of
// 961 scores 7.0 us (now 4.1), 189 of 3974 20 (6.2), 517 of 2053 22 (6.7), 3844 of 961 24 (12), 3844 of 4000 78 (32): scores of
// prompt chunks, a token's rows visible up to its position. (3844 of 961 with all rows visible 13.8, Gaussian scores 15.9.)
constexpr uint32_t kRowBins = 1024;
constexpr uint32_t kNegInfKey = 0x007FFFFFu;

template <int OFF>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, OFF, 0xF, 0xF, false);
}
__device__ __forceinline__ uint32_t umax(uint32_t a, uint32_t b) { return a > b ? a : b; }
__device__ __forceinline__ uint32_t umin(uint32_t a, uint32_t b) { return a < b ? a : b; }
// maximum over the wave, in every lane
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
  v = umax(v, dpp_u32<0x128>(v));  // row_ror:8
  v = umax(v, dpp_u32<0x124>(v));  // row_ror:4
  v = umax(v, dpp_u32<0x122>(v));  // row_ror:2
  v = umax(v, dpp_u32<0x121>(v));  // row_ror:1
  uint32_t r = (uint32_t)__builtin_amdgcn_readlane((int)v, 0);
  r = umax(r, (uint32_t)__builtin_amdgcn_readlane((int)v, 16));
  r = umax(r, (uint32_t)__builtin_amdgcn_readlane((int)v, 32));
  return umax(r, (uint32_t)__builtin_amdgcn_readlane((int)v, 48));
}

template <int C, int THREADS>
__global__ __launch_bounds__(THREADS) void topk_row_kernel(const float* __restrict__ scores_all, int64_t score_stride,
                                                           int n_rows, int topk, int32_t* __restrict__ sel_all) {
  constexpr int kW = THREADS / 64;
  static_assert(C <= 32 && kRowBins % THREADS == 0, "a lane per chunk, whole zeroing rounds");
  __shared__ __attribute__((aligned(16))) uint32_t hist[kRowBins];
  __shared__ __attribute__((aligned(16))) uint32_t cnt[C * kW];  // hits per (chunk, wave): above low, ties high
  __shared__ uint32_t red_max[kW], red_not_low[kW], red_count[kW];
  __shared__ uint32_t list[64];
  __shared__ uint32_t list_n;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const float* scores = scores_all + (int64_t)blockIdx.x * score_stride;
  int32_t* sel = sel_all + (int64_t)blockIdx.x * topk;

  // (All requested at once, past the end the last score again: under a condition each load is waited for before the next. One row
  // of 961 scores 4.16 -> 3.56 us, 15 rows of 2015 5.9 -> 4.2, 3844 rows of 961 12.2 -> 11.3.)
  float score[C];
#pragma unroll
  for (int j = 0; j < C; j++) {
    const int e = j * THREADS + tid;
    score[j] = scores[e < n_rows ? e : n_rows - 1];
  }
  uint32_t key[C];
#pragma unroll
  for (int j = 0; j < C; j++) key[j] = j * THREADS + tid < n_rows ? score_key(score[j]) : 0u;
#pragma unroll
  for (int i = 0; i < (int)kRowBins / THREADS; i++) hist[i * THREADS + tid] = 0u;
  if (tid == 0) list_n = 0u;
  uint32_t top4[4] = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int j = 0; j < C; j++) top4[j & 3] = umax(key[j], top4[j & 3]);
  const uint32_t even = umax(top4[0], top4[2]), odd = umax(top4[1], top4[3]);
  uint32_t hi = umax(even, odd);
  // the lowest of the maxima of disjoint groups of keys, of which there are at least k, is not above the k-th key
  const uint32_t group = topk <= THREADS ? hi : topk <= 2 * THREADS ? umin(even, odd) :
                         topk <= 4 * THREADS ? umin(umin(top4[0], top4[1]), umin(top4[2], top4[3])) : 0u;
  hi = wave_max(hi);
  const uint32_t not_bound = wave_max(~group);
  if (lane == 0) {
    red_max[wave] = hi;
    red_not_low[wave] = not_bound;
  }
  __syncthreads();
  hi = wave_max(red_max[lane % kW]);
  uint32_t lo = ~wave_max(red_not_low[lane % kW]);

  uint32_t need = (uint32_t)topk, threshold = kNegInfKey;
  bool found = false;
  if (lo <= kNegInfKey) {  // not bounded by finite groups: the lowest finite key, or what lies below
    uint32_t not_low = 0u, n_fin = 0u, n_inf = 0u;
#pragma unroll
    for (int j = 0; j < C; j++) {
      const bool fin = key[j] > kNegInfKey;
      not_low = umax(fin ? ~key[j] : 0u, not_low);
      n_fin += (uint32_t)__popcll(__ballot(fin));
      n_inf += (uint32_t)__popcll(__ballot(key[j] == kNegInfKey));
    }
    not_low = wave_max(not_low);
    __syncthreads();  // every wave has read the bounds
    if (lane == 0) {
      red_not_low[wave] = not_low;
      red_count[wave] = n_fin | (n_inf << 16);
    }
    __syncthreads();
    lo = ~wave_max(red_not_low[lane % kW]);
    const uint32_t counts = (uint32_t)__builtin_amdgcn_readlane((int)wave_prefix_sum(lane < kW ? red_count[lane] : 0u), 63);
    n_fin = counts & 0xFFFFu;
    n_inf = counts >> 16;
    if (need > n_fin) {  // the k-th key is -inf, or one of the negative NaNs below it
      need -= n_fin;
      found = need <= n_inf;
      if (!found) need -= n_inf;
      lo = 0u;
      hi = kNegInfKey - 1u;
    }
  }
  uint32_t span = hi - lo;
  while (!found) {
    const int shift = span >= kRowBins ? 22 - __builtin_clz(span) : 0;
#pragma unroll
    for (int j = 0; j < C; j++) {
      const uint32_t d = key[j] - lo;
      if (d <= span) atomicAdd(&hist[d >> shift], 1u);
    }
    __syncthreads();
    // lane l holds the sixteen bins below 1024 - 16 l, so that a prefix sum over lanes counts from the top
    uint32_t t[16];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(&hist[16 * (63 - lane) + 4 * i]);
#pragma unroll
      for (int c = 0; c < 4; c++) t[4 * i + c] = v[c];
    }
    uint32_t sum = 0u;
#pragma unroll
    for (int i = 0; i < 16; i++) sum += t[i];
    const uint32_t incl = wave_prefix_sum(sum);
    uint32_t run = incl - sum, left = 0u, held = 0u, bin = 0u;
#pragma unroll
    for (int i = 15; i >= 0; i--) {
      const bool here = run < need && run + t[i] >= need;
      bin = here ? (uint32_t)(16 * (63 - lane) + i) : bin;
      left = here ? need - run : left;
      held = here ? t[i] : held;
      run += t[i];
    }
    const int src = (int)__builtin_ctzll(__ballot(held != 0u));
    bin = (uint32_t)__builtin_amdgcn_readlane((int)bin, src);
    need = (uint32_t)__builtin_amdgcn_readlane((int)left, src);
    held = (uint32_t)__builtin_amdgcn_readlane((int)held, src);
    lo += bin << shift;
    const uint32_t rest = span - (bin << shift), width = (1u << shift) - 1u;
    span = rest < width ? rest : width;
    if (span == 0u) {
      threshold = lo;
      break;
    }
    if (held <= 64u) {
#pragma unroll
      for (int j = 0; j < C; j++) {
        const bool in = key[j] - lo <= span;
        if (in) list[atomicAdd(&list_n, 1u)] = key[j];
      }
      __syncthreads();
      const uint32_t mine = list[lane];
      uint32_t above = 0u, ties = 0u;
      for (int i = 0; i < (int)held; i++) {
        const uint32_t o = (uint32_t)__builtin_amdgcn_readlane((int)mine, i);
        above += o > mine ? 1u : 0u;
        ties += o == mine ? 1u : 0u;
      }
      const int at = (int)__builtin_ctzll(__ballot(lane < (int)held && above < need && above + ties >= need));
      threshold = (uint32_t)__builtin_amdgcn_readlane((int)mine, at);
      need -= (uint32_t)__builtin_amdgcn_readlane((int)above, at);
      break;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < (int)kRowBins / THREADS; i++) hist[i * THREADS + tid] = 0u;
    __syncthreads();
  }
  const uint32_t n_above = (uint32_t)topk - need;

  uint32_t hits = 0u;
#pragma unroll
  for (int j = 0; j < C; j++) {
    const uint32_t a = (uint32_t)__popcll(__ballot(key[j] > threshold)), t = (uint32_t)__popcll(__ballot(key[j] == threshold));
    hits = lane == j ? a | (t << 16) : hits;
  }
  if (lane < C) cnt[lane * kW + wave] = hits;
  __syncthreads();
  uint32_t row_sum = 0u, before = 0u;  // of chunk `lane`: all waves, the waves in front of this one
  if (lane < C) {
#pragma unroll
    for (int w = 0; w < kW; w++) {
      const uint32_t c = cnt[lane * kW + w];
      row_sum += c;
      before += w < wave ? c : 0u;
    }
  }
  before += wave_prefix_sum(row_sum) - row_sum;
  asm volatile("" : "+s"(threshold));  // the votes below are taken again, not kept in 4 C scalar registers
#pragma unroll
  for (int j = 0; j < C; j++) {
    const uint32_t base = (uint32_t)__builtin_amdgcn_readlane((int)before, j);
    const bool above = key[j] > threshold, tie = key[j] == threshold;
    const uint64_t ba = __ballot(above), bt = __ballot(tie);
    const uint32_t ra = __builtin_amdgcn_mbcnt_hi((uint32_t)(ba >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)ba, base & 0xFFFFu));
    if (above) sel[ra] = j * THREADS + tid;
    if (bt != 0ull) {
      const uint32_t rt = __builtin_amdgcn_mbcnt_hi((uint32_t)(bt >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bt, base >> 16));
      if (tie && rt < need) sel[n_above + rt] = j * THREADS + tid;
    }
  }
}

// Rows of up to 4 P THREADS scores, one a workgroup, where k is a small part of them: what is done per key is one comparison
// with a pivot that lies below the k-th key nearly always, and the rest is done on the keys at or above it.
//  * Every wave takes 64 S keys spread over the row and finds the 16-bit prefix of the `rank`-th of them with ballots; the
//    mean of the waves' prefixes is the pivot. One barrier, no histogram.
//  * The rows at or above it go to a list in LDS, in any order; their keys are read from a copy of the row in LDS. Where they are
//    fewer than k, the list is made again from the lowest of the waves' prefixes: a wave samples stretches of the row, and of
//    a row whose scores change along it the mean may say nothing (97 % of the wanted scores in one stretch: 1 row of 32768, k =
//    2048, 42 us through the binning of all keys, now 13.7; 3844 of 8192, k = 512, 144 and 45). Where all parts are alike it is
//    one row in some hundreds, which the launch then waits for: 3844 rows of 7961 Gaussian scores 33.5 us, now 26.
//  * 256 bins over [pivot, highest sample] hold the k-th key; a bin of up to 64 keys (nearly always the first one) is ranked
//    directly, otherwise it becomes the span.
//  * Selected rows set their bit in a bitmap of the row. Bits come out in row order, so nothing before has to keep it.
// Keys are compared as signed integers: the bits of a float32 themselves where the pivot is positive, all others after the
// map that inverts the low bits of negative values. Whether the list contains the k-th key is checked exactly; if it does not
// (or does not fit, or a second round of bins hardly splits it), the binning runs over all keys, so the result never depends
// on the sample. There -inf is counted on the side, the span is that of the keys in question, and votes go to copies of the
// counters: in one histogram the votes of a row that is mostly -inf, or of one value, follow each other on one counter in
// every pass (1 row of 32768, k = 2048, 400 finite: 125 us, now 13; 3844 rows of 8192, k = 512, 100 finite: 484, now 44; a
// chunk of 8400 tokens from position 0, whose first quarter sees too few rows: scores selected in 100, now 37).
// What bounds it: a CU takes 2000 cycles to fetch a row of 32768 scores, and an instruction per key is 500 cycles of its vector
// units: the blocked kernel above maps and moves every key (two LDS passes) and takes five digit passes, 16 rows of 32768,
// k = 2048, 10.0 us, now 7.7. For many rows it is instructions: 3844 rows of 7961, k = 512, 57 us, now 26. (Keys read again
// from the L2 instead of from a copy of the row in LDS: 64 lines an instruction, 3 us more for 16 rows; neighbouring lanes on
// neighbouring list entries: their bits meet in the same words, 1 us more.)
constexpr int32_t kLowestKey = (int32_t)0x80000000u;
constexpr int32_t kNegInfSigned = (int32_t)(kNegInfKey ^ 0x80000000u);

__device__ __forceinline__ int32_t signed_key(int32_t bits) { return bits ^ (int32_t)((uint32_t)(bits >> 31) >> 1); }

// mask = 16 mask + (bits k.w, k.z, k.y, k.x at or above the pivot): a comparison and an addition with carry a key. (From the
// compiler it is four instructions and two wait states: a comparison's result may not be read by the next two. With the list
// written two rows at a time, the sample read from the copy of the row, its end shifted instead of loaded again and only the
// waves with a candidate ranking one: 16 rows of 32768 scores, k = 2048, 8.4 -> 7.7 us; 3844 of 7961, k = 512, 29.4 -> 26.2; 5 of
// 19211, k = 1024, 7.2 -> 6.8; 1 of 4096, k = 512, 4.6 and 4.6. The pivot is taken from a vector register: in a scalar one that a
// vector instruction has just written, the first comparison would be one of those two, and the compiler puts no wait states in
// front of inline assembly. Within it, three instructions lie between a comparison and the addition that reads it.)
__device__ __forceinline__ uint32_t shift_in_four(uint32_t mask, __attribute__((ext_vector_type(4))) int k, int32_t pivot) {
  uint64_t c0, c1, c2, c3;
  asm("v_cmp_le_i32_e64 %1, %9, %5\n\tv_cmp_le_i32_e64 %2, %9, %6\n\tv_cmp_le_i32_e64 %3, %9, %7\n\t"
      "v_cmp_le_i32_e64 %4, %9, %8\n\t"
      "v_addc_co_u32_e64 %0, vcc, %0, %0, %1\n\tv_addc_co_u32_e64 %0, vcc, %0, %0, %2\n\t"
      "v_addc_co_u32_e64 %0, vcc, %0, %0, %3\n\tv_addc_co_u32_e64 %0, vcc, %0, %0, %4"
      : "+v"(mask), "=&s"(c0), "=&s"(c1), "=&s"(c2), "=&s"(c3)
      : "v"(k.w), "v"(k.z), "v"(k.y), "v"(k.x), "v"(pivot)
      : "vcc");
  return mask;
}

template <int P, int THREADS, int S>
__global__ __launch_bounds__(THREADS) void topk_sampled_kernel(const float* __restrict__ scores_all, int64_t score_stride,
                                                               int n_rows, int topk, int rank,
                                                               int32_t* __restrict__ sel_all) {
  constexpr int kW = THREADS / 64;
  constexpr int kEach = 8;                 // list entries of a thread at most
  constexpr int kCap = kEach * THREADS;
  constexpr uint32_t kBits = 4 * P;        // of the bitmap, to a word: a word a thread
  constexpr uint32_t kBins = 256;
  static_assert(kBits <= 32 && S <= P && kBins <= THREADS && 16 % kW == 0, "a bin a thread, a piece a sample");
  __shared__ __attribute__((aligned(16))) int32_t stage[4 * P * THREADS];
  __shared__ __attribute__((aligned(16))) uint16_t list[kCap];
  __shared__ __attribute__((aligned(16))) uint32_t hist[kBins];
  __shared__ uint32_t bits_above[THREADS], bits_tie[THREADS];
  __shared__ uint32_t wave_pivot[kW], wave_high[kW];
  __shared__ uint32_t wave_tot[kW];
  __shared__ __attribute__((aligned(16))) uint32_t near[64];
  __shared__ uint32_t kth[2];
  __shared__ Pick pick_box;
  __shared__ uint32_t n_list[2], n_near;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const float* scores = scores_all + (int64_t)blockIdx.x * score_stride;
  int32_t* sel = sel_all + (int64_t)blockIdx.x * topk;

  // ---- keys: element e of piece j of a thread is row 4 (j THREADS + tid) + e; past the end the lowest key, which loses every
  //      tie to a real row. (Rows start at any multiple of 4 bytes.)
  typedef __attribute__((ext_vector_type(4), aligned(4))) int i32x4_any_t;
  typedef __attribute__((ext_vector_type(4))) int i32x4_t;
  auto row_of = [&](int j, int e) { return 4 * (j * THREADS + tid) + e; };
  i32x4_t key[P];
  const int last_four = n_rows - 4;  // (n_rows is at least 4)
#pragma unroll
  for (int j = 0; j < P; j++) {
    const int r = row_of(j, 0);
    key[j] = *reinterpret_cast<const i32x4_any_t*>(scores + (r < last_four ? r : last_four));
  }
  if (tid < (int)kBins) hist[tid] = 0u;
  bits_above[tid] = 0u;
  bits_tie[tid] = 0u;
  if (tid == 0) {
    n_list[0] = 0u;
    n_list[1] = 0u;
    n_near = 0u;
  }
#pragma unroll
  for (int j = 0; j < P; j++) {
    const int r = row_of(j, 0);
    if (4 * (j + 1) * THREADS > n_rows) {  // (uniform: pieces in front of the row's end are whole)
      // the row's last four scores, shifted (loaded one by one, they held up everything behind them)
      const int by = r - last_four;
      i32x4_t k = key[j];
      if (by > 0 && (by & 1)) k = i32x4_t{k.y, k.z, k.w, -1};
      if (by > 0 && (by & 2)) k = i32x4_t{k.z, k.w, -1, -1};
      if (by > 3) k = i32x4_t{-1, -1, -1, -1};
      key[j] = k;
    }
    *reinterpret_cast<i32x4_t*>(&stage[r]) = key[j];
  }

  // ---- this wave's sample: lane l takes element l / P % 4 of pieces l + i of the P
  uint32_t sample[S];
  uint32_t high = 0u;
#pragma unroll
  for (int i = 0; i < S; i++) {
    const int piece = (lane + i) % P, e = (lane / P) & 3;
    int32_t v = 0;
    if constexpr (P > 2) {
      v = stage[row_of(piece, e)];  // (its own copy: picked by comparison it is five instructions a piece)
    } else {
#pragma unroll
      for (int j = 0; j < P; j++) {
        const i32x4_t k = key[j];
        const int32_t x = e & 2 ? (e & 1 ? k.w : k.z) : (e & 1 ? k.y : k.x);
        v = piece == j ? x : v;
      }
    }
    sample[i] = (uint32_t)signed_key(v) ^ 0x80000000u;
    high = umax(high, sample[i]);
  }
  high = wave_max(high);
  uint32_t prefix = 0u;
#pragma unroll
  for (int bit = 31; bit >= 16; bit--) {
    const uint32_t with = prefix | (1u << bit);
    int n = 0;
#pragma unroll
    for (int i = 0; i < S; i++) n += (int)__popcll(__ballot(sample[i] >= with));
    prefix = n >= rank ? with : prefix;
  }
  if (lane == 0) {
    wave_pivot[wave] = prefix >> 16;
    wave_high[wave] = high;
  }
  __syncthreads();
  int32_t pivot, span_end;
  bool masked;  // the wanted rank of some wave's sample is -inf (or below)
  {
    uint32_t sum = wave_pivot[lane % kW], top = wave_high[lane % kW];  // (the same sixteen values in every row of lanes)
    masked = __ballot(sum <= kNegInfKey >> 16) != 0ull;
    sum += dpp_u32<0x128>(sum);
    sum += dpp_u32<0x124>(sum);
    sum += dpp_u32<0x122>(sum);
    sum += dpp_u32<0x121>(sum);
    top = umax(top, dpp_u32<0x128>(top));
    top = umax(top, dpp_u32<0x124>(top));
    top = umax(top, dpp_u32<0x122>(top));
    top = umax(top, dpp_u32<0x121>(top));
    pivot = __builtin_amdgcn_readfirstlane((int)(((sum >> 4) << 16) ^ 0x80000000u));
    span_end = __builtin_amdgcn_readfirstlane((int)(top ^ 0x80000000u));
  }
  auto uniform = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };

  // ---- rows at or above the pivot
  bool mapped = false;
  auto listed = [&](uint32_t* counter) -> uint32_t {
    if (!mapped && pivot <= 0) {  // uniform
      mapped = true;
#pragma unroll
      for (int j = 0; j < P; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) key[j][e] = signed_key(key[j][e]);
    }
    uint32_t mask = 0u;
#pragma unroll
    for (int j = P - 1; j >= 0; j--) mask = shift_in_four(mask, key[j], pivot);
    const uint32_t cnt = (uint32_t)__popc(mask);
    const uint32_t incl = wave_prefix_sum(cnt);
    uint32_t base = 0u;
    if (lane == 63) base = atomicAdd(counter, incl);
    base = (uint32_t)__builtin_amdgcn_readlane((int)base, 63);
    if (base + (uint32_t)__builtin_amdgcn_readlane((int)incl, 63) <= (uint32_t)kCap) {
      uint16_t* at = list + base + incl - cnt;
      auto row_of_bit = [&](int i) { return (uint16_t)row_of(i >> 2, i & 3); };
      while (mask) {  // (two at a time, where a thread has many; a last odd one is written twice)
        const int i = __builtin_ctz(mask);
        mask &= mask - 1u;
        if constexpr (P < 4) {
          *at++ = row_of_bit(i);
          continue;
        }
        const uint32_t another = mask != 0u ? 1u : 0u;
        const int i2 = another ? __builtin_ctz(mask) : i;
        at[0] = row_of_bit(i);
        at[another] = row_of_bit(i2);
        at += 2;
        mask &= mask - 1u;
      }
    }
    __syncthreads();
    return uniform(*counter);
  };
  // (One at or below -inf would list the rows a token does not see as well: those are counted below, not binned. Where the
  // waves' parts of the row differ, the mean of their pivots may lie above the k-th key: the lowest of them is taken then.)
  uint32_t total = 0u;
  if (pivot > kNegInfSigned) {  // uniform
    total = listed(&n_list[0]);
    if (__builtin_expect(total < (uint32_t)topk && !masked, 0)) {
      pivot = (int32_t)((uniform(~wave_max(~wave_pivot[lane % kW])) << 16) ^ 0x80000000u);
      total = listed(&n_list[1]);
    }
  }
  const bool fits = total >= (uint32_t)topk && total <= (uint32_t)kCap;  // uniform

  // ---- the k-th key, k = need, is one of those in [lo, lo + limit]; `span` is a guess of the distance from lo to the highest
  //      one (what is above is in the last bin)
  uint32_t need = (uint32_t)topk, limit = 0xFFFFFFFFu, span;
  int32_t lo = pivot, threshold = 0;
  bool found = fits;
  // of the votes in `hist`, 1 << shift keys wide a bin: the bin with the k-th key, and how many keys it holds
  auto narrow = [&](int shift) -> uint32_t {
    __syncthreads();
    Pick pk;
    if constexpr (kW <= 4) {
      pk = pick_bucket(hist, need, lane);  // (every wave for itself: handed on by one, it was a barrier and a read more)
    } else {  // (four waves a SIMD wait for each other's instructions longer than that)
      if (wave == 0) {
        pk = pick_bucket(hist, need, lane);
        if (lane == 0) pick_box = pk;
      }
      __syncthreads();
      pk = Pick{uniform(pick_box.digit), uniform(pick_box.need), uniform(pick_box.live)};
    }
    const uint32_t bin = pk.digit;
    need = pk.need;
    lo = (int32_t)((uint32_t)lo + (bin << shift));
    const uint32_t rest = limit - (bin << shift), width = bin == kBins - 1u ? 0xFFFFFFFFu : (1u << shift) - 1u;
    limit = rest < width ? rest : width;
    return pk.live;
  };
  auto candidate = [&](int32_t k) {
    const bool in = k >= lo && (uint32_t)k - (uint32_t)lo <= limit;
    if (__ballot(in) != 0ull) {  // (few waves hold any)
      if (in) near[atomicAdd(&n_near, 1u)] = (uint32_t)k - (uint32_t)lo;
    }
  };
  // the k-th of up to 64 candidates: sixteen lanes rank one, each against four at a time
  auto rank_candidates = [&](uint32_t held) {
    __syncthreads();
    constexpr int kAtOnce = THREADS / 16;
#pragma unroll
    for (int c0 = 0; c0 < 64; c0 += kAtOnce) {
      if ((uint32_t)(c0 + 4 * wave) >= held) break;  // (the wave's four)
      const int c = c0 + (tid >> 4);
      const uint32_t mine = near[c];
      const u32x4_t o = *reinterpret_cast<const u32x4_t*>(&near[4 * (lane & 15)]);
      uint32_t n = 0u;  // higher ones, equal ones in the upper half
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const bool in = (uint32_t)(4 * (lane & 15) + j) < held;
        n += in && o[j] > mine ? 1u : 0u;
        n += in && o[j] == mine ? 1u << 16 : 0u;
      }
      n += dpp_u32<0x128>(n);
      n += dpp_u32<0x124>(n);
      n += dpp_u32<0x122>(n);
      n += dpp_u32<0x121>(n);
      const uint32_t above = n & 0xFFFFu;
      if ((lane & 15) == 0 && (uint32_t)c < held && above < need && above + (n >> 16) >= need) {  // (all equal ones write the same)
        kth[0] = mine;
        kth[1] = need - above;
      }
    }
    __syncthreads();
    need = uniform(kth[1]);
    lo = (int32_t)((uint32_t)lo + uniform(kth[0]));
    limit = 0u;
  };

  if (fits) {
    constexpr int kHalf = kEach / 2;
    int32_t lk[kEach];
    int lr[kEach];
    const bool more = total > (uint32_t)(kHalf * THREADS);  // uniform
    // (entry j of a thread: neighbouring lanes take entries a wave count apart, whose rows are in different bitmap words)
    const uint32_t first = (uint32_t)(lane * kW + wave);
    auto fetch = [&](int j0) {
#pragma unroll
      for (int j = j0; j < j0 + kHalf; j++) lr[j] = (int)list[j * THREADS + first];
#pragma unroll
      for (int j = j0; j < j0 + kHalf; j++) lr[j] = (uint32_t)(j * THREADS) + first < total ? lr[j] : 0;
#pragma unroll
      for (int j = j0; j < j0 + kHalf; j++) lk[j] = stage[lr[j]];
#pragma unroll
      for (int j = j0; j < j0 + kHalf; j++) {
        if (mapped) lk[j] = signed_key(lk[j]);
        lk[j] = (uint32_t)(j * THREADS) + first < total ? lk[j] : kLowestKey;
      }
    };
    fetch(0);
    if (more) fetch(kHalf);
    auto each = [&](auto f) {
#pragma unroll
      for (int j = 0; j < kHalf; j++) f(lk[j], lr[j]);
      if (more) {
#pragma unroll
        for (int j = kHalf; j < kEach; j++) f(lk[j], lr[j]);
      }
    };
    if (__builtin_expect(masked, 0)) {  // (uniform) a mean with -inf in it lies far below the listed keys: the lowest of them
      uint32_t not_low = 0u;
      each([&](int32_t k, int) { not_low = umax(not_low, k != kLowestKey ? ~((uint32_t)k ^ 0x80000000u) : 0u); });
      not_low = wave_max(not_low);
      if (lane == 0) wave_pivot[wave] = not_low;
      __syncthreads();
      lo = (int32_t)(uniform(~wave_max(wave_pivot[lane % kW])) ^ 0x80000000u);
    }
    span = span_end > lo ? (uint32_t)span_end - (uint32_t)lo : 0u;
    uint32_t half = 0xFFFFFFFFu;  // of the keys that the bin before held
    while (true) {
      const int shift = span >= kBins ? 24 - __builtin_clz(span) : 0;
      each([&](int32_t k, int) {
        const uint32_t d = (uint32_t)k - (uint32_t)lo;
        if (k >= lo && d <= limit) atomicAdd(&hist[umin(d >> shift, kBins - 1u)], 1u);
      });
      const uint32_t held = narrow(shift);
      if (limit == 0u) break;
      if (held <= 64u) {
        each([&](int32_t k, int) { candidate(k); });
        rank_candidates(held);
        break;
      }
      if (held > 512u && held > half) {  // keys that meet in one bin again and again
        found = false;
        break;
      }
      span = limit;
      half = held / 2u;
      __syncthreads();  // every wave has read the counters
      if (tid < (int)kBins) hist[tid] = 0u;
      __syncthreads();
    }
    if (found) {
      threshold = lo;
      each([&](int32_t k, int row) {
        const uint32_t word = (uint32_t)row / kBits, bit = 1u << ((uint32_t)row % kBits);
        if (k > threshold) atomicOr(&bits_above[word], bit);
        if (k == threshold) atomicOr(&bits_tie[word], bit);
      });
    }
  }
  if (__builtin_expect(!found, 0)) {
    // All keys, from the copy of the row: rows with fewer finite scores than are wanted, rows of few values, and where the
    // sample misled.
    auto each = [&](auto f) {
#pragma unroll 2
      for (int j = 0; j < P; j++) {
        i32x4_t k = *reinterpret_cast<const i32x4_t*>(&stage[4 * (j * THREADS + tid)]);
#pragma unroll
        for (int e = 0; e < 4; e++) k[e] = signed_key(k[e]);
        f(k, 4u * (uint32_t)(j * THREADS + tid));
      }
    };
    limit = umin(limit, 0x7FFFFFFFu - (uint32_t)lo);
    if (!fits) {
      // The bins are those of the keys above -inf, or at the pivot and above where the list overflowed. Those of -inf are counted:
      // rows a token does not see yet are most of a row at the start of a prompt, and the k-th key is -inf where fewer are seen
      // than are wanted.
      const int32_t low = total > (uint32_t)kCap ? pivot : kNegInfSigned + 1;
      uint32_t not_low = 0u, top = 0u, counts = 0u;  // lowest of them, highest key, how many and how many of -inf
      each([&](i32x4_t k, uint32_t) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const uint32_t u = (uint32_t)k[e] ^ 0x80000000u;
          const bool in = k[e] >= low;
          top = umax(top, u);
          not_low = umax(not_low, in ? ~u : 0u);
          counts += in ? 1u : k[e] == kNegInfSigned ? 1u << 16 : 0u;
        }
      });
      top = wave_max(top);
      not_low = wave_max(not_low);
      counts = wave_prefix_sum(counts);
      __syncthreads();  // every wave has read the pivots
      if (lane == 63) {
        wave_pivot[wave] = not_low;
        wave_high[wave] = top;
        wave_tot[wave] = counts;
      }
      __syncthreads();
      lo = (int32_t)(uniform(~wave_max(wave_pivot[lane % kW])) ^ 0x80000000u);
      int32_t end = (int32_t)(uniform(wave_max(wave_high[lane % kW])) ^ 0x80000000u);
      counts = (uint32_t)__builtin_amdgcn_readlane((int)wave_prefix_sum(lane < kW ? wave_tot[lane % kW] : 0u), 63);
      const uint32_t n_in = counts & 0xFFFFu, n_inf = counts >> 16;
      if (need > n_in) {  // -inf, or one of the negative NaNs below it
        need -= n_in;
        lo = end = kNegInfSigned;
        if (need > n_inf) {
          need -= n_inf;
          lo = kLowestKey;
          end = kNegInfSigned - 1;
        }
      }
      limit = (uint32_t)end - (uint32_t)lo;
    }
    while (limit != 0u) {
      // votes go to kCopies copies of the counters, which take the list's place, so that few of a wave's meet
      constexpr int kVoteCopies = kCap / 2 / (int)kBins, kPerBin = THREADS / (int)kBins;
      static_assert(kVoteCopies == 4 * kPerBin, "a thread adds four copies");
      uint32_t* counters = reinterpret_cast<uint32_t*>(list);
      *reinterpret_cast<u32x4_t*>(&counters[4 * tid]) = u32x4_t{0u, 0u, 0u, 0u};
      __syncthreads();
      const int shift = limit >= kBins ? 24 - __builtin_clz(limit) : 0;
      each([&](i32x4_t k, uint32_t) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const uint32_t d = (uint32_t)k[e] - (uint32_t)lo;
          if (d <= limit)  // (keys below lo are further off than any above it)
            atomicAdd(&counters[(d >> shift) * kVoteCopies + (uint32_t)(lane % kVoteCopies)], 1u);
        }
      });
      __syncthreads();
      const u32x4_t c = *reinterpret_cast<const u32x4_t*>(&counters[4 * tid]);  // kPerBin neighbouring lanes have a bin
      uint32_t sum = c.x + c.y + c.z + c.w;
#pragma unroll
      for (int m = 1; m < kPerBin; m *= 2) sum += __shfl_xor(sum, m, MSPR_WAVE);
      if (tid % kPerBin == 0) hist[tid / kPerBin] = sum;
      const uint32_t held = narrow(shift);
      if (limit != 0u && held <= 64u) {
        each([&](i32x4_t k, uint32_t) {
#pragma unroll
          for (int e = 0; e < 4; e++) candidate(k[e]);
        });
        rank_candidates(held);
      }
    }
    threshold = lo;
    // the four rows of a piece are in one word of the bitmap
    each([&](i32x4_t k, uint32_t row) {
      uint32_t above = 0u, tie = 0u;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        above |= k[e] > threshold ? 1u << e : 0u;
        tie |= k[e] == threshold ? 1u << e : 0u;
      }
      if (above != 0u) atomicOr(&bits_above[row / kBits], above << (row % kBits));
      if (tie != 0u) atomicOr(&bits_tie[row / kBits], tie << (row % kBits));
    });
  }
  __syncthreads();

  // ---- the selected rows
  uint32_t wa = bits_above[tid], wt = bits_tie[tid];
  const uint32_t mine = (uint32_t)__popc(wa) | ((uint32_t)__popc(wt) << 16);
  const uint32_t upto = wave_prefix_sum(mine);
  if (lane == 63) wave_tot[wave] = upto;
  __syncthreads();
  const uint32_t tots = wave_prefix_sum(lane < kW ? wave_tot[lane < kW ? lane : 0] : 0u);
  const uint32_t excl = upto - mine + (wave > 0 ? (uint32_t)__builtin_amdgcn_readlane((int)tots, wave > 0 ? wave - 1 : 0) : 0u);
  int32_t* out = sel + (excl & 0xFFFFu);
  uint32_t order = excl >> 16;
  while (wa) {
    *out++ = (int)kBits * tid + (int)__builtin_ctz(wa);
    wa &= wa - 1u;
  }
  out = sel + ((uint32_t)topk - need);
  while (wt && order < need) {
    out[order++] = (int)kBits * tid + (int)__builtin_ctz(wt);
    wt &= wt - 1u;
  }
}

// Rank of the pivot in a wave's 64 S keys: as many as are expected above the k-th key of the (padded) row, and 3 standard
// deviations of the mean of the waves' ranks on top. 0 where the keys above such a pivot would not fit the list.
int sample_rank(int keys, int waves, int s, int cap, int topk) {
  const double share = (double)topk / keys, n = 64.0 * s, expect = share * n;
  const double dev = std::sqrt((expect > 1.0 ? expect : 1.0) * (1.0 - share) / waves);
  const double rank = std::ceil(expect + 3.0 * dev + 0.5);
  if (rank > n || (rank + 4.0 * dev) / n * keys > (double)cap) return 0;
  return (int)rank;
}

// Rank, inside the 1024-row sample, of the pivot of the pivot path; 0 switches the path off. With k of
// the C*1024 (padded) rows wanted, k/C sample rows are expected above the k-th key; the rank adds 4.5
// standard deviations so that the survivors almost always include it, and the path is used only where
// the survivors then almost always (6 more deviations) fit the list. A miss on either side costs time,
// not correctness: the kernel checks the survivor count and falls back to the full passes.
int pivot_sample_rank(int c, int topk) {
  const double expect = (double)topk / c;
  const double rank = std::ceil(expect + 4.5 * std::sqrt(expect) + 2.0);
  const double worst = rank * c + 6.0 * c * std::sqrt(rank);
  if (rank > 512.0 || worst > (double)kFastCap) return 0;
  return (int)rank;
}

}  // namespace

int mspr_launch_topk(const float* scores, int64_t score_stride, int batch, int64_t n_rows, int topk, int32_t* sel,
                     hipStream_t st) {
  dim3 grid((unsigned)batch), block(kThreads);
  MsprProfScope prof(MSPR_K_TOPK, st);
  // Rows of more than 2048 scores of which at most three eighths (past 4096: less than a half) are wanted are selected from the
  // keys above a sampled pivot, where those fit its list: 512 threads a row, 256 where many rows share the CUs, 1024 for what
  // only they can hold. us, the other kernels and this one: 1 row of 4096 scores, k = 512, 5.3 and 4.6; of 8192, k = 2048, 7.2
  // and 6.1; 5 of 19211, k = 1024, 9.3 and 6.8; 16 of 32768, k = 2048, 10.0 and 7.7; 517 of 7000, k = 512, 10.5 and 7.0; 3844 of
  // 3000 24.5 and 18.2, of 7961 57 and 26; 600 of 16384 27 and 19. At the lines: 4096 scores 1 row, k = 1500, 5.7 and 5.4, k =
  // 2048 5.5 and 6.3; 2100 scores, k = 700, 1 row 4.9 and 5.1, 517 7.0 and 6.6; 1500 scores, k = 512, 4.5 and 4.9, 3844 rows 16.2
  // and 16.4; 8192 scores, k = 3000, 7.5 and 7.3, k = 4000 7.6 and 9.1. 384 rows of 4096, k = 512: 512 threads 6.4, 256 6.0; 256
  // rows 5.4 and 5.6.
  if (n_rows > 2048 && n_rows <= 32768 && (n_rows <= 4096 ? 8 * (int64_t)topk <= 3 * n_rows : 2 * (int64_t)topk < n_rows)) {
    auto pieces = [&](int threads) { return (int)((n_rows + 4 * threads - 1) / (4 * threads)); };
    int p = 0, threads = 0, rank = 0;
    if (n_rows > 8192) {
      p = pieces(threads = 1024) == 7 ? 8 : pieces(1024);
      rank = sample_rank(4 * 1024 * p, 16, 1, 8 * 1024, topk);
    } else {
      if (batch > 384) {
        p = pieces(threads = 256) == 7 ? 8 : pieces(256);
        rank = sample_rank(4 * 256 * p, 4, 2, 8 * 256, topk);
      }
      if (rank == 0) {
        p = pieces(threads = 512);
        rank = sample_rank(4 * 512 * p, 8, 2, 8 * 512, topk);
      }
    }
#define MSPR_TOPK_SAMPLED(P, THREADS, S)                                                                                      \
  if (rank > 0 && p == P && threads == THREADS) {                                                                             \
    topk_sampled_kernel<P, THREADS, S><<<grid, dim3(THREADS), 0, st>>>(scores, score_stride, (int)n_rows, topk, rank, sel);    \
    MSPR_CHECK_LAUNCH("topk_select");                                                                                         \
    return MSPR_OK;                                                                                                           \
  }
    MSPR_TOPK_SAMPLED(3, 256, 2)
    MSPR_TOPK_SAMPLED(4, 256, 2)
    MSPR_TOPK_SAMPLED(5, 256, 2)
    MSPR_TOPK_SAMPLED(6, 256, 2)
    MSPR_TOPK_SAMPLED(8, 256, 2)
    MSPR_TOPK_SAMPLED(2, 512, 2)
    MSPR_TOPK_SAMPLED(3, 512, 2)
    MSPR_TOPK_SAMPLED(4, 512, 2)
    MSPR_TOPK_SAMPLED(3, 1024, 1)
    MSPR_TOPK_SAMPLED(4, 1024, 1)
    MSPR_TOPK_SAMPLED(5, 1024, 1)
    MSPR_TOPK_SAMPLED(6, 1024, 1)
    MSPR_TOPK_SAMPLED(8, 1024, 1)
#undef MSPR_TOPK_SAMPLED
  }
  // The others. Up to 4096 scores a row: 256 threads a row keep the most rows in flight; a row of more than 2048 that has a CU
  // for itself is better off with 512. Up to 8192 many rows take the row kernel too, few take the blocked form, whose sample
  // bounds a large k better; past that its work per key is less.
#define MSPR_TOPK_ROW(C, THREADS) \
  topk_row_kernel<C, THREADS><<<grid, dim3(THREADS), 0, st>>>(scores, score_stride, (int)n_rows, topk, sel)
  if (n_rows <= 1024) MSPR_TOPK_ROW(4, 256);
  else if (n_rows <= 2048) MSPR_TOPK_ROW(8, 256);
  else if (n_rows <= 4096 && batch <= 256) MSPR_TOPK_ROW(8, 512);
  else if (n_rows <= 3072) MSPR_TOPK_ROW(12, 256);
  else if (n_rows <= 4096) MSPR_TOPK_ROW(16, 256);
  else if (n_rows <= 8192 && batch > 32) MSPR_TOPK_ROW(16, 512);
#undef MSPR_TOPK_ROW
  else if (n_rows <= 8 * 1024)
    topk_blocked_kernel<8, true><<<grid, block, 0, st>>>(scores, score_stride, (int)n_rows, topk, pivot_sample_rank(8, topk), sel);
  else if (n_rows <= 32 * 1024)
    topk_blocked_kernel<32, false><<<grid, block, 0, st>>>(scores, score_stride, (int)n_rows, topk, 0, sel);
  else topk_select_kernel<<<grid, block, 0, st>>>(scores, score_stride, n_rows, topk, sel);
  MSPR_CHECK_LAUNCH("topk_select");
  return MSPR_OK;
}

extern "C" int mspr_topk_select(const float* scores, int64_t score_stride, int batch, int64_t n_rows, int topk,
                                int32_t* sel, void* stream) {
  MSPR_REQUIRE(scores && sel, "topk_select: null pointer");
  MSPR_REQUIRE(batch >= 1, "topk_select: batch must be positive");
  MSPR_REQUIRE(n_rows >= 1 && n_rows < (int64_t)1 << 31, "topk_select: n_rows must be in [1, 2^31)");
  MSPR_REQUIRE(topk >= 1 && topk <= n_rows, "topk_select: topk must be positive and at most n_rows");
  MSPR_REQUIRE(score_stride >= n_rows, "topk_select: score_stride must cover a row");
  return mspr_launch_topk(scores, score_stride, batch, n_rows, topk, sel, (hipStream_t)stream);
}
