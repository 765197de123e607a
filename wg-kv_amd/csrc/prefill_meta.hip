// Vertical-slash metadata of the sparse prefill (gfx950), built on the device.
//
// Replaces generate_sparse_indices / generate_block_offset /
// generate_column_index (src/modeling_layers.py:321-409), which loop over
// (batch, head) on the host with a torch.nonzero and a .item() sync each.
//
// Count blocks: block 0 is position 0 alone, block k >= 1 covers
// [1 + (k-1)*bs, 1 + k*bs) -- the grouping whose running sums give, for row
// block r >= P, the number of admitted positions below r*bs - W + 1.  Block k
// thus ends at position k*bs, and column_count[k + P] is the inclusive count
// there; the listed range is [0, (R-1)*bs].
//
// A workgroup takes `span` consecutive tiles of one (b, h).  It counts the
// flags before its first tile itself (16 per load, an L2 read after the first
// workgroup), so no workgroup waits for another and one launch does it all; then
// thread t takes positions t, t + 256, ... of a tile, a ballot ranks a wave's
// 64 flags and one scan over the tile's (step, wave) counts places them.  The
// reads before the tiles grow with the square of the prompt, so long prompts
// take larger tiles and then more of them per workgroup.  Bound by latency (a
// few memory round trips): one workgroup per head walking 64-flag blocks byte
// by byte took 22 us at 9001 tokens and 17 us at 777 (8 heads), launched back
// to back; this takes 3.8 and 3.2 us.  The workgroups after the last head's
// write the band tables, which depend only on (W, S, bs).
#include <type_traits>

#include "wgkv_common.h"

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kShortList = 196608;  // listed positions up to this take 1024-position tiles
constexpr int kMaxWgs = 512;        // workgroups per (b, h) at most

struct MetaArgs {
  const uint8_t* mask;
  int64_t m_sb, m_sh;
  int B, H, S, W, bs, R, P;
  int32_t* block_count;
  int32_t* block_offset;
  int32_t* column_count;
  int32_t* column_index;
  int col_cap;
  int32_t* column_total;
  int wgs;   // workgroups per (b, h)
  int span;  // tiles per workgroup
};

template <int STEPS>  // 256-position steps per tile
__global__ __launch_bounds__(kThreads) void prefill_meta_kernel(MetaArgs a) {
  __shared__ int s_pre[kWaves];
  __shared__ int s_cnt[STEPS * kWaves];
  const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
  constexpr unsigned kStep = STEPS * kThreads;
  const int bh = blockIdx.x / a.wgs, wg = blockIdx.x - bh * a.wgs;
  if (bh == a.B * a.H) {
    // band tables (one row per row block, P+1 entries each)
    const int width = a.P + 1;
    const int last_first = max(0, (a.R - 1) * a.bs - a.W + 1);
    const int last_count = (a.S - last_first + a.bs - 1) / a.bs;
    const int64_t stride = (int64_t)a.wgs * kThreads;
    for (int64_t e = (int64_t)wg * kThreads + t; e < (int64_t)a.R * width; e += stride) {
      const int r = (int)(e / width), c = (int)(e - (int64_t)r * width);
      a.block_offset[e] = r < a.P ? (c < a.P ? c * a.bs : 0) : 1 + (r - a.P + c) * a.bs;
      if (c == 0) a.block_count[r] = r == a.R - 1 ? last_count : r < a.P ? r + 1 : width;
    }
    return;
  }
  const int b = bh / a.H, h = bh - b * a.H;
  const uint8_t* m = a.mask + (int64_t)b * a.m_sb + (int64_t)h * a.m_sh;
  int32_t* cc = a.column_count + (int64_t)bh * a.R;
  int32_t* ci = a.column_index + (int64_t)bh * a.col_cap;
  // positions unsigned: the last tile may reach past 2^31
  const unsigned n_list = (unsigned)(a.R - 1) * a.bs + 1;
  const unsigned begin = wg * (STEPS == 4 ? 1 : a.span) * kStep;
  if (wg == 0)
    for (int r = t; r < min(a.P, a.R); r += kThreads) cc[r] = 0;

  int run = 0;  // admitted before the wave's 64 flags of the step
  const auto take = [&](unsigned p0, auto first) {
    // this tile's flags, and for the first one the count before it
    uint64_t bal[STEPS];
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      const unsigned p = p0 + i * kThreads + t;
      bal[i] = __builtin_amdgcn_ballot_w64(p < n_list && m[p] != 0);
    }
    int pre = 0;
    if constexpr (first) pre = wave_sum_int(count_flags(m, 0, (int)p0, t, kThreads));
    else __syncthreads();  // the last tile's counts are read
    if (lane == 0) {
      if (first) s_pre[wid] = pre;
#pragma unroll
      for (int i = 0; i < STEPS; ++i) s_cnt[i * kWaves + wid] = __builtin_popcountll(bal[i]);
    }
    __syncthreads();
    if (first) run = (s_pre[0] + s_pre[1]) + (s_pre[2] + s_pre[3]);
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      int mine = run;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const int c = s_cnt[i * kWaves + w];
        mine += w < wid ? c : 0;
        run += c;
      }
      const unsigned p = p0 + i * kThreads + t;
      const bool f = bal[i] >> lane & 1;
      const int rank = mine + __builtin_popcountll(bal[i] & ((1ull << lane) - 1));
      if (f && rank < a.col_cap) ci[rank] = (int)p;
      if (p < n_list && p % a.bs == 0) {
        const int64_t r = (int64_t)(p / a.bs) + a.P;
        if (r < a.R) cc[r] = rank + (f ? 1 : 0);
      }
    }
  };
  take(begin, std::true_type{});
  const unsigned span = STEPS == 4 ? 1 : a.span;  // short prompts: one tile
  if (span > 1)
    for (unsigned p0 = begin + kStep; p0 < min(n_list, begin + span * kStep); p0 += kStep) take(p0, std::false_type{});
  if (t == 0 && a.column_total && n_list - begin <= span * kStep) a.column_total[bh] = run;
}

}  // namespace

extern "C" int wgkv_build_prefill_meta(
    const uint8_t* g_mask, int64_t gm_stride_b, int64_t gm_stride_h,
    int32_t batch, int32_t num_kv_heads, int32_t seq_len, int32_t local_window, int32_t block,
    int32_t* block_count, int32_t* block_offset,
    int32_t* column_count, int32_t* column_index, int32_t col_cap, int32_t* column_total,
    void* stream) {
  if (!g_mask || !block_count || !block_offset || !column_count || !column_index) return WGKV_ERR_ARG;
  if (batch <= 0 || num_kv_heads <= 0 || seq_len <= 0 || block <= 0 || local_window < 0 || col_cap < 0)
    return WGKV_ERR_ARG;
  if (local_window % block) return WGKV_ERR_ARG;  // the reference asserts W % bs == 0
  MetaArgs a;
  a.mask = g_mask;
  a.m_sb = gm_stride_b;
  a.m_sh = gm_stride_h;
  a.B = batch;
  a.H = num_kv_heads;
  a.S = seq_len;
  a.W = local_window;
  a.bs = block;
  a.R = (seq_len + block - 1) / block;
  a.P = min(local_window / block, a.R);
  a.block_count = block_count;
  a.block_offset = block_offset;
  a.column_count = column_count;
  a.column_index = column_index;
  a.col_cap = col_cap;
  a.column_total = column_total;
  // Positions per workgroup: 1024 while the flags before a tile are read by few
  // loads per thread, 4096 where those reads outweigh the tile's own work.  8
  // heads, 1024 / 4096: 65536 positions 6.6 / 10.1 us, 131072 9.9 / 12.9,
  // 262144 25.7 / 18.6, 400000 37.9 / 24.8.  Past kMaxWgs tiles a workgroup takes
  // several, so that the reads before them grow with the prompt and not with
  // its square: 8 heads, one tile / span tiles: 4 million positions 660 / 410 us,
  // 16 million 14.9 / 2.6 ms; one head of 100 million 142 / 3.4 ms.
  const int n_list = (a.R - 1) * block + 1;
  const int tile = n_list <= kShortList ? 1024 : 4096;
  const int tiles = n_list / tile + (n_list % tile != 0);
  a.span = (tiles + kMaxWgs - 1) / kMaxWgs;
  a.wgs = (tiles + a.span - 1) / a.span;
  const dim3 grid((unsigned)a.wgs * (batch * num_kv_heads + 1));
  if (tile == 1024)
    hipLaunchKernelGGL(prefill_meta_kernel<4>, grid, dim3(kThreads), 0, (hipStream_t)stream, a);
  else
    hipLaunchKernelGGL(prefill_meta_kernel<16>, grid, dim3(kThreads), 0, (hipStream_t)stream, a);
  return hipGetLastError() == hipSuccess ? WGKV_OK : WGKV_ERR_HIP;
}
