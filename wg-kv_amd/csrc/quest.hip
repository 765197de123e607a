// QUEST page selection over the dual cache's page tables (gfx950).
//
// The reference's comparison baseline (src/modeling_layers.py:452-576 with
// the page bounds kept at :1333-1347 and :744-761): every global page keeps
// the elementwise min and max of its keys; at a decode step each head scores
// its full global pages by max over the grouped queries of
// sum_d q_d * (q_d >= 0 ? max_d : min_d), keeps the top pages within a token
// budget (after its local window), always keeps the trailing partial page,
// and the decode attention runs over the local pages plus the kept pages.
//
//   * quest_bounds_kernel: recompute the bounds of a head's logical global
//     pages [from/page, ceil(len/page)) from the pool (the min / max over the
//     page's valid rows, which equals the reference's incremental updates);
//   * quest_scores_kernel: the page scores of every head into the workspace;
//   * quest_select_kernel: one workgroup per head -- the k-th largest score
//     by bisection of its bits, then a stable compaction that writes local
//     pages, the kept full pages in page order and the partial page, and the
//     head's token count.
// Scores are fp32, or (scores_bf16) rounded as the reference's bf16 torch ops
// round them: each product q_d * bound_d to bf16, the fp32 sum over d to
// bf16.  Equal scores at the cut keep the lowest page index (the reference's
// topk leaves their order unspecified).
#include "wgkv_common.h"

namespace {

constexpr int kThreads = 256;

struct BoundsArgs {
  const uint16_t* pool_k;
  const int32_t* bt;  // block_table + layer * H * max_pages
  int max_pages, lb;  // pages per head, local pages per head
  const int32_t* len;   // global_lengths + layer * H
  const int32_t* from;  // global lengths before the update (NULL: 0)
  int H, page, D;
  uint16_t* kmin;
  uint16_t* kmax;
};

__device__ __forceinline__ float bf(uint16_t x) { return __uint_as_float((uint32_t)x << 16); }
__device__ __forceinline__ float round_bf16f(float x) { return round_to_bf16(x); }

// grid (H, groups): workgroup g of head h takes pages first+g, first+g+groups, ...
__global__ __launch_bounds__(kThreads) void quest_bounds_kernel(BoundsArgs a) {
  const int h = blockIdx.x;
  const int n = a.len[h];
  const int f = a.from ? a.from[h] : 0;
  const int first = f / a.page, last = (n + a.page - 1) / a.page;  // [first, last)
  const int32_t* bt = a.bt + (int64_t)h * a.max_pages + a.lb;
  const int per = kThreads / a.D;  // pages per pass (D <= 256)
  const int sub = threadIdx.x / a.D, d = threadIdx.x % a.D;
  if (sub >= per) return;
  for (int p = first + blockIdx.y * per + sub; p < last; p += gridDim.y * per) {
    const int rows = min(a.page, n - p * a.page);
    const int64_t pg = bt[p];
    const uint16_t* src = a.pool_k + pg * a.page * a.D + d;
    uint16_t lo = src[0], hi = src[0];
    for (int r = 1; r < rows; ++r) {
      const uint16_t x = src[(int64_t)r * a.D];
      if (bf(x) < bf(lo)) lo = x;
      if (bf(x) > bf(hi)) hi = x;
    }
    a.kmin[pg * a.D + d] = lo;
    a.kmax[pg * a.D + d] = hi;
  }
}

struct SelectArgs {
  const uint16_t* q;  // (Hq, D) of this token, stride q_sh
  int64_t q_sh;
  const int32_t* bt;   // block_table + layer * H * max_pages
  int max_pages, lb;
  const int32_t* len;  // global_lengths + layer * H
  const uint16_t* kmin;
  const uint16_t* kmax;
  int H, D, page, local_tokens, scores_bf16;
  int local_blocks, budget_blocks;  // pages of the local tokens and of the budget past them
  int32_t* sel_bt;     // (H, sel_cap)
  int sel_cap;
  int32_t* sel_len;    // (H)
  float* scores;       // workspace (H, max_pages)
};

// Page scores: 16 lanes per page, 8 d-values each (16-byte loads of the
// bounds and, from LDS, of the group members' queries), summed per lane in d
// order and then over the 16 lanes; workgroups stride over the head's full
// pages, two of them per lane group in flight.  Bound by latency
// (a 128K prompt's 13.1K pages are 6.7 MB of bounds): the group size is a
// template argument, as a runtime bound put the per-member sums in scratch
// memory and read the queries from LDS value by value (30.2 us, median of a
// trace; now 6.8).
template <int G, bool BF16>
__global__ __launch_bounds__(kThreads) void quest_scores_kernel(SelectArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t s_q[G][256];
  const int h = blockIdx.y, t = threadIdx.x;
  const int full = a.len[h] / a.page;
  if ((int)blockIdx.x * 16 >= full) return;
  for (int e = t; e < G * a.D; e += kThreads) {
    const int g = e / a.D, d = e - g * a.D;
    s_q[g][d] = a.q[(int64_t)(h * G + g) * a.q_sh + d];
  }
  __syncthreads();
  const int32_t* bt = a.bt + (int64_t)h * a.max_pages + a.lb;
  float* sc = a.scores + (int64_t)h * a.max_pages;
  const int lane16 = t & 15, slot = t >> 4;  // 16 pages per pass
  const int nch = a.D / 8;                   // 8-value chunks per row (<= 32)
  constexpr int U = 2;                       // passes in flight
  const int step = gridDim.x * 16;
  for (int p0 = blockIdx.x * 16 + slot; p0 < full + slot; p0 += step * U) {
    int64_t row[U];
    bool ok[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      ok[u] = p0 + u * step < full;
      row[u] = (int64_t)bt[ok[u] ? p0 + u * step : 0] * a.D;
    }
    float s[U][G] = {};
    for (int c = lane16; c < nch; c += 16) {
      u32x4_t lo[U], hi[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        lo[u] = *(const u32x4_t*)(a.kmin + row[u] + c * 8);
        hi[u] = *(const u32x4_t*)(a.kmax + row[u] + c * 8);
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const u32x4_t qv = *(const u32x4_t*)&s_q[g][c * 8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float q0 = bf16lo(qv[e]), q1 = bf16hi(qv[e]);
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const float b0 = q0 >= 0.f ? bf16lo(hi[u][e]) : bf16lo(lo[u][e]);
            const float b1 = q1 >= 0.f ? bf16hi(hi[u][e]) : bf16hi(lo[u][e]);
            // a product of two bf16 values is exact in fp32; bf16 ops round it
            if (BF16) {
              const uint32_t r = pack_bf16x2(q0 * b0, q1 * b1);
              s[u][g] = (s[u][g] + bf16lo(r)) + bf16hi(r);
            } else {
              s[u][g] = fmaf(q1, b1, fmaf(q0, b0, s[u][g]));
            }
          }
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float best = -INFINITY;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const float v = row_sum16(s[u][g]);
        best = fmaxf(best, BF16 ? round_bf16f(v) : v);
      }
      if (ok[u] && lane16 == 0) sc[p0 + u * step] = best;
    }
  }
}

// order-preserving map of an fp32 to uint32 (larger float -> larger key)
__device__ __forceinline__ uint32_t fkey(float f) {
  const uint32_t u = __float_as_uint(f);
  return u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
}

// Largest / smallest of x over the wave (DPP within rows of 16, then scalar).
__device__ __forceinline__ uint32_t wave_umax(uint32_t x) {
  x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, WGKV_DPP_QP_1032, 0xf, 0xf, false));
  x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, WGKV_DPP_QP_2301, 0xf, 0xf, false));
  x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, WGKV_DPP_ROW_HALF_MIRROR, 0xf, 0xf, false));
  x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, WGKV_DPP_ROW_MIRROR, 0xf, 0xf, false));
  const uint32_t a = max((uint32_t)__builtin_amdgcn_readlane((int)x, 0), (uint32_t)__builtin_amdgcn_readlane((int)x, 16));
  const uint32_t b = max((uint32_t)__builtin_amdgcn_readlane((int)x, 32), (uint32_t)__builtin_amdgcn_readlane((int)x, 48));
  return max(a, b);
}

// The selection of a head's `keep` largest of `full` page scores (0 < keep <
// full) by one workgroup, kept pages written in page order from out on.  The
// keep-th largest key T is found two bits at a time -- the largest T with at
// least `keep` keys >= T -- with counts from ballots: no histogram, whose
// bins the equal exponents of page scores crowd into.  A step takes ~1100
// cycles.  The leading bits that all keys share need no step, so scores of one
// sign leave the exponent's out and scores of both signs leave out none.
// Scores rounded to bf16 differ only in the key's upper half: at most 8 steps,
// 4 or 5 where the scores have one sign.  fp32 scores would take up to 16, but
// rarely tie: they stop once exactly `keep` keys reach T, after some log2(full)
// bits below the shared ones (8 heads of 1638 pages, G 4, scores and selection
// 15.2 us with all steps, 13.0 with the stop; with bf16 scores, which tie, the
// test costs 0.3 of 12.6 us and is left out).  With STAGED the keys are read
// once and kept in LDS (heads of up to kMaxKeys pages), else the scores are
// read again in every step.
constexpr int kMaxKeys = 12288;  // a multiple of 8 * kThreads
constexpr int kWaves = kThreads / 64;
constexpr int kRows = 8;  // rows of kThreads pages handled together

template <bool BF16, bool STAGED>
__device__ void select_pages(const float* sc, int full, int keep, const int32_t* pages, int32_t* out,
                             uint32_t* s_key, int (*s_cnt)[3][kWaves], int* s_pref) {
  constexpr int BITS = BF16 ? 16 : 32;
  const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
  const int rows = (full + kThreads - 1) / kThreads;  // of kThreads pages
  // key of page p, 0 past the head's pages: below every tested value
  auto read_key = [&](int p) {
    const uint32_t x = fkey(sc[min(p, full - 1)]) >> (32 - BITS);
    return p < full ? x : 0u;
  };
  auto key_at = [&](int p) { return STAGED ? s_key[p] : read_key(p); };
  // whole groups of rows; each thread reads back only its own keys: no barrier
  uint32_t hi = 0, lo = 0;  // the largest key, and the largest complement of one
  for (int r0 = 0; r0 < rows; r0 += kRows) {
    uint32_t x[kRows];
#pragma unroll
    for (int j = 0; j < kRows; ++j) x[j] = read_key((r0 + j) * kThreads + t);
#pragma unroll
    for (int j = 0; j < kRows; ++j) {
      const int p = (r0 + j) * kThreads + t;
      if (STAGED) s_key[p] = x[j];
      hi = max(hi, x[j]);
      lo = max(lo, p < full ? ~x[j] : 0u);
    }
  }
  hi = wave_umax(hi);
  lo = wave_umax(lo);
  if (lane == 0) {
    s_pref[wid] = (int)hi;
    s_pref[kWaves + wid] = (int)lo;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    hi = max(hi, (uint32_t)s_pref[w]);
    lo = max(lo, (uint32_t)s_pref[kWaves + w]);
  }
  const uint32_t diff = hi ^ ~lo;  // the bits in which the largest and the smallest key differ
  const int top = diff ? (33 - __builtin_clz(diff)) & ~1 : 0;  // an even number of low bits that holds them
  uint32_t T = top < 32 ? hi >> top << top : 0u;
  T = __builtin_amdgcn_readfirstlane(T);
  int above = 0;  // keys >= T's last tested successor: keys > T at the end
#pragma unroll 1
  for (int shift = __builtin_amdgcn_readfirstlane(top) - 2, step = 0; shift >= 0; shift -= 2, step ^= 1) {
    int c[3] = {0, 0, 0};
#pragma unroll 1
    for (int r0 = 0; r0 < rows; r0 += kRows) {
      uint32_t x[kRows];
#pragma unroll
      for (int j = 0; j < kRows; ++j) x[j] = key_at((r0 + j) * kThreads + t);
#pragma unroll
      for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int j = 0; j < kRows; ++j)
          c[d] += __builtin_popcountll(__builtin_amdgcn_ballot_w64(x[j] >= (T | ((uint32_t)(d + 1) << shift))));
    }
    // a step's counts are read before the next step's barrier: two sets suffice
#pragma unroll
    for (int d = 0; d < 3; ++d)
      if (lane == 0) s_cnt[step][d][wid] = c[d];
    __syncthreads();
#pragma unroll
    for (int d = 0; d < 3; ++d)
      c[d] = (s_cnt[step][d][0] + s_cnt[step][d][1]) + (s_cnt[step][d][2] + s_cnt[step][d][3]);
    const int digit = c[2] >= keep ? 3 : c[1] >= keep ? 2 : c[0] >= keep ? 1 : 0;
    T = __builtin_amdgcn_readfirstlane(T | (uint32_t)digit << shift);
    if (digit < 3) above = c[digit];
    if constexpr (!BF16) {
      const int reached = digit == 3 ? c[2] : digit == 2 ? c[1] : c[0];  // keys >= the new T (digit > 0)
      if (digit > 0 && reached == keep) {  // exactly the kept keys: no lower bit matters
        --T;
        above = keep;
        break;
      }
    }
  }
  // kept: key > T, plus the first need_eq pages (in page order) with key ==
  // T.  kRows rows at a time: each (row, wave)'s two counts packed in one word,
  // their prefix in page order, then the kept pages' places; the page ids are
  // requested first.
  const int need_eq = keep - above;
  int base_gt = 0, base_eq = 0;  // before the group (a group's own counts fit 16 bits)
  for (int r0 = 0; r0 < rows; r0 += kRows) {
    int32_t id[kRows];
    uint64_t gt[kRows], eq[kRows];
#pragma unroll
    for (int j = 0; j < kRows; ++j) id[j] = pages[min((r0 + j) * kThreads + t, full - 1)];
    __syncthreads();  // s_pref is free
#pragma unroll
    for (int j = 0; j < kRows; ++j) {
      const int p = (r0 + j) * kThreads + t;
      const uint32_t x = key_at(p);
      gt[j] = __builtin_amdgcn_ballot_w64(x > T);
      eq[j] = __builtin_amdgcn_ballot_w64(x == T && p < full);
      if (lane == 0) s_pref[j * kWaves + wid] = __builtin_popcountll(gt[j]) << 16 | __builtin_popcountll(eq[j]);
    }
    __syncthreads();
    const int mine = lane < kRows * kWaves ? s_pref[lane] : 0;
    const int incl = wave_incl_scan(mine, lane);
    const uint64_t below = (1ull << lane) - 1;
#pragma unroll
    for (int j = 0; j < kRows; ++j) {
      const int before = __builtin_amdgcn_readlane(incl - mine, __builtin_amdgcn_readfirstlane(j * kWaves + wid));
      const int rank_gt = base_gt + (before >> 16) + __builtin_popcountll(gt[j] & below);
      const int rank_eq = base_eq + (before & 0xffff) + __builtin_popcountll(eq[j] & below);
      if ((gt[j] >> lane & 1) || ((eq[j] >> lane & 1) && rank_eq < need_eq)) out[rank_gt + min(rank_eq, need_eq)] = id[j];
    }
    const int total = __builtin_amdgcn_readlane(incl, 63);
    base_gt += total >> 16;
    base_eq += total & 0xffff;
  }
}

// The same for a head of at most kThreads pages, a page per thread: a page is
// kept if fewer than `keep` pages rank before it (a larger key, or the same
// key and an earlier page).  One pass over the keys takes less than the steps
// above for few pages (kFewPages, kFewPagesBf16): scores and selection of 8
// heads, G 4, steps / this: fp32 scores of 100 pages 10.4 / 7.7 us, of 200
// 10.5 / 10.0; bf16 scores of 60 pages 9.9 / 7.3, of 100 9.9 / 8.1, of 200
// 10.0 / 10.3.
constexpr int kFewPages = kThreads, kFewPagesBf16 = 160;

__device__ void select_few_pages(const float* sc, int full, int keep, const int32_t* pages, int32_t* out,
                                 uint32_t* s_key, int* s_pref) {
  const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
  const int p = min(t, full - 1);
  const int32_t id = pages[p];
  const uint32_t x = fkey(sc[p]);
  s_key[t] = t < full ? x : 0u;  // below every page's key
  __syncthreads();
  int rank = 0;
  for (int q = 0; q < full; q += 4) {
    const u32x4_t v = *(const u32x4_t*)(s_key + q);
#pragma unroll
    for (int e = 0; e < 4; ++e) rank += v[e] > x || (v[e] == x && q + e < t);
  }
  const uint64_t kept = __builtin_amdgcn_ballot_w64(t < full && rank < keep);
  if (lane == 0) s_pref[wid] = __builtin_popcountll(kept);
  __syncthreads();
  int at = __builtin_popcountll(kept & ((1ull << lane) - 1));
#pragma unroll
  for (int w = 0; w < kWaves; ++w) at += w < wid ? s_pref[w] : 0;
  if (kept >> lane & 1) out[at] = id;
}

// One workgroup per head.  Bound by latency (a few memory round trips and the
// steps' barriers); four waves rather than sixteen, whose barriers and scalar
// counting cost more than the keys.  1638 pages per head, 8 heads, bf16 scores,
// medians of a trace: 14.7 us with four LDS-histogram passes over the scores in
// memory, 9.0 us in this form.
template <bool BF16>
__global__ __launch_bounds__(kThreads) void quest_select_kernel(SelectArgs a) {
  __shared__ __attribute__((aligned(16))) uint32_t s_key[kMaxKeys];
  __shared__ int s_cnt[2][3][kWaves];
  __shared__ int s_pref[kRows * kWaves];
  const int h = blockIdx.x, t = threadIdx.x;
  const int32_t* bt = a.bt + (int64_t)h * a.max_pages;
  int32_t* out = a.sel_bt + (int64_t)h * a.sel_cap;
  const float* sc = a.scores + (int64_t)h * a.max_pages;
  const int n = a.len[h];
  const int local_blocks = a.local_blocks;
  for (int i = t; i < local_blocks; i += kThreads) out[i] = bt[i];
  const int full = n / a.page, rem = n - full * a.page;
  const int capacity = min(a.budget_blocks, full + (rem > 0 ? 1 : 0));
  const bool partial = capacity > 0 && rem > 0;
  const int k = capacity - (rem > 0 ? 1 : 0);  // full pages to keep
  const bool all = k >= full;
  const int keep = k <= 0 ? 0 : (all ? full : k);
  if (keep > 0 && !all) {
    if (full <= (BF16 ? kFewPagesBf16 : kFewPages))
      select_few_pages(sc, full, keep, bt + a.lb, out + local_blocks, s_key, s_pref);
    else if (full <= kMaxKeys)
      select_pages<BF16, true>(sc, full, keep, bt + a.lb, out + local_blocks, s_key, s_cnt, s_pref);
    else
      select_pages<BF16, false>(sc, full, keep, bt + a.lb, out + local_blocks, s_key, s_cnt, s_pref);
  } else if (keep > 0) {
    for (int p = t; p < keep; p += kThreads) out[local_blocks + p] = bt[a.lb + p];
  }
  if (t == 0) {
    if (partial) out[local_blocks + keep] = bt[a.lb + full];
    a.sel_len[h] = a.local_tokens + keep * a.page + (partial ? rem : 0);
  }
}

template <int G>
void launch_select(const SelectArgs& a, hipStream_t st) {
  // a head's pages over at least 64 workgroups, the call over about 1024; no
  // more than its table could fill
  const int most = (a.max_pages - a.lb + 15) / 16, want = max(64, 1024 / a.H);
  const dim3 grid(max(1, min(most, want)), a.H);
  if (a.scores_bf16) {
    hipLaunchKernelGGL((quest_scores_kernel<G, true>), grid, dim3(kThreads), 0, st, a);
    hipLaunchKernelGGL(quest_select_kernel<true>, dim3(a.H), dim3(kThreads), 0, st, a);
  } else {
    hipLaunchKernelGGL((quest_scores_kernel<G, false>), grid, dim3(kThreads), 0, st, a);
    hipLaunchKernelGGL(quest_select_kernel<false>, dim3(a.H), dim3(kThreads), 0, st, a);
  }
}

}  // namespace

extern "C" int wgkv_quest_update_bounds(
    const void* pool_k, const int32_t* block_table, int32_t max_pages_per_head,
    const int32_t* global_lengths, const int32_t* from_lengths,
    int32_t layer, int32_t num_layers, int32_t num_kv_heads, int32_t local_window, int32_t page_size,
    int32_t head_dim, void* key_min, void* key_max, void* stream) {
  if (!pool_k || !block_table || !global_lengths || !key_min || !key_max) return WGKV_ERR_ARG;
  if (layer < 0 || layer >= num_layers || num_kv_heads <= 0 || page_size <= 0 || local_window % page_size)
    return WGKV_ERR_ARG;
  if (head_dim <= 0 || head_dim > kThreads || kThreads % head_dim) return WGKV_ERR_UNSUPPORTED;
  BoundsArgs a;
  a.pool_k = (const uint16_t*)pool_k;
  a.bt = block_table + (int64_t)layer * num_kv_heads * max_pages_per_head;
  a.max_pages = max_pages_per_head;
  a.lb = local_window / page_size;
  a.len = global_lengths + (int64_t)layer * num_kv_heads;
  a.from = from_lengths;
  a.H = num_kv_heads;
  a.page = page_size;
  a.D = head_dim;
  a.kmin = (uint16_t*)key_min;
  a.kmax = (uint16_t*)key_max;
  hipLaunchKernelGGL(quest_bounds_kernel, dim3(num_kv_heads, 64), dim3(kThreads), 0, (hipStream_t)stream, a);
  return hipGetLastError() == hipSuccess ? WGKV_OK : WGKV_ERR_HIP;
}

extern "C" size_t wgkv_quest_select_workspace_bytes(int32_t num_kv_heads, int32_t max_pages_per_head) {
  return (size_t)num_kv_heads * max_pages_per_head * sizeof(float);
}

extern "C" int wgkv_quest_select(
    const void* q, int64_t q_stride_h,
    const int32_t* block_table, int32_t max_pages_per_head, const int32_t* global_lengths,
    const void* key_min, const void* key_max,
    int32_t layer, int32_t num_layers, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
    int32_t local_window, int32_t page_size, int32_t local_tokens, int32_t token_budget, int32_t scores_bf16,
    int32_t* sel_block_table, int32_t sel_cap, int32_t* sel_seqlens,
    void* workspace, size_t workspace_bytes, void* stream) {
  if (!q || !block_table || !global_lengths || !key_min || !key_max || !sel_block_table || !sel_seqlens)
    return WGKV_ERR_ARG;
  if (layer < 0 || layer >= num_layers || num_kv_heads <= 0 || num_q_heads % num_kv_heads) return WGKV_ERR_ARG;
  if (page_size <= 0 || local_window % page_size || local_tokens < 0 || local_tokens > local_window) return WGKV_ERR_ARG;
  const int G = num_q_heads / num_kv_heads;
  if (G > 8 || head_dim <= 0 || head_dim > 256 || head_dim % 8) return WGKV_ERR_UNSUPPORTED;
  if (((uintptr_t)key_min | (uintptr_t)key_max) & 15) return WGKV_ERR_UNSUPPORTED;
  const int local_blocks = (local_tokens + page_size - 1) / page_size;
  const int budget_blocks = ((token_budget > local_tokens ? token_budget - local_tokens : 0) + page_size - 1) / page_size;
  if (sel_cap < local_blocks + budget_blocks) return WGKV_ERR_ARG;
  if (!workspace || workspace_bytes < wgkv_quest_select_workspace_bytes(num_kv_heads, max_pages_per_head))
    return WGKV_ERR_WORKSPACE;
  SelectArgs a;
  a.q = (const uint16_t*)q;
  a.q_sh = q_stride_h;
  a.bt = block_table + (int64_t)layer * num_kv_heads * max_pages_per_head;
  a.max_pages = max_pages_per_head;
  a.lb = local_window / page_size;
  a.len = global_lengths + (int64_t)layer * num_kv_heads;
  a.kmin = (const uint16_t*)key_min;
  a.kmax = (const uint16_t*)key_max;
  a.H = num_kv_heads;
  a.D = head_dim;
  a.page = page_size;
  a.local_tokens = local_tokens;
  a.local_blocks = local_blocks;
  a.budget_blocks = budget_blocks;
  a.scores_bf16 = scores_bf16 ? 1 : 0;
  a.sel_bt = sel_block_table;
  a.sel_cap = sel_cap;
  a.sel_len = sel_seqlens;
  a.scores = (float*)workspace;
  hipStream_t st = (hipStream_t)stream;
  switch (G) {
    case 1: launch_select<1>(a, st); break;
    case 2: launch_select<2>(a, st); break;
    case 3: launch_select<3>(a, st); break;
    case 4: launch_select<4>(a, st); break;
    case 5: launch_select<5>(a, st); break;
    case 6: launch_select<6>(a, st); break;
    case 7: launch_select<7>(a, st); break;
    default: launch_select<8>(a, st); break;
  }
  return hipGetLastError() == hipSuccess ? WGKV_OK : WGKV_ERR_HIP;
}
