// Chunked gated prefill: cache writes around the attention of one chunk
// (gfx950).  The reference prefills the whole prompt at once
// (src/modeling_layers.py:1183-1376); a chunk [c0, c0+C) here leaves the dual
// cache exactly as a one-shot prefill of the first c0+C tokens would, up to
// page numbering:
//   * admit: the admitted positions of [c0-W, c0+C-W) -- the previous ring
//     (slot i holds position c0-W+i, flag in local_is_global) followed by the
//     chunk -- are appended in position order to each head's global cache
//     (so it stays sorted), new pages bump-allocated in head order as a head
//     crosses page boundaries;
//   * column_count of the chunk's row blocks = admitted positions below
//     max(0, r*64 - W + 1): the global length before the chunk plus a prefix
//     count over (ring flags ++ chunk mask);
//   * ring (after the chunk's attention): slot i <- position c0+C-W+i.
// Requires, for every chunk after the first, c0 >= W (a full ring) and C >= W
// (the ring then refills from the chunk alone); c0 and W multiples of 64.
#include "wgkv_common.h"

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kBlk = 64;      // virtual positions per scatter step
constexpr int kMaxSpan = 8;   // steps per workgroup at most

struct ChunkArgs {
  const uint16_t* key;
  const uint16_t* value;
  int64_t kv_sh, kv_ss;
  const uint16_t* pre_key;
  int64_t pk_sh, pk_ss;
  const uint8_t* mask;  // chunk flags (H, C)
  int64_t m_sh;
  int layer, H, C, D, W, page, max_tokens_per_head, c0;
  int64_t total_pages;
  uint16_t* pool_k;
  uint16_t* pool_v;
  int32_t* block_table;
  int max_pages;
  int32_t* global_lengths;
  uint8_t* local_is_global;
  uint16_t* local_pre_key;
  int32_t* next_free;
  int32_t* status;
  int32_t* column_count;  // (H, R_chunk)
  int r0, rchunk;         // first global row block of the chunk, row blocks in the chunk
  int span;               // 64-position steps per admission workgroup
  int lph;                // lanes that count a head's flags: 64, 16, 4 or 1
  // workspace, written by stage 0 and read by stage 1
  int32_t* adm;           // (H) positions admitted by the chunk
  int32_t* gl_before;     // (H) global lengths before the chunk
  int32_t* next_free_after;
  int32_t* abort_flag;
};

constexpr int kMaxHeads = 1024;

// Virtual sequence of a chunk: ring positions (c0 > 0 only) then the chunk.
__host__ __device__ __forceinline__ int vlen(const ChunkArgs& a) { return (a.c0 > 0 ? a.W : 0) + a.C; }
__host__ __device__ __forceinline__ int vring(const ChunkArgs& a) { return a.c0 > 0 ? a.W : 0; }

// Admitted flags of head h among the first n virtual positions, this thread's
// share (t of nt threads).
__device__ __forceinline__ int vcount(const ChunkArgs& a, int h, int n, int t, int nt) {
  const int nr = vring(a);
  int c = count_flags(a.mask + (int64_t)h * a.m_sh, 0, n - nr, t, nt);
  if (nr > 0) c += count_flags(a.local_is_global + ((int64_t)a.layer * a.H + h) * a.W, 0, min(nr, n), t, nt);
  return c;
}

// Admission of one chunk in one launch (workgroup = `span` steps of 64
// virtual positions of one head).  Every workgroup first counts the admitted
// flags of every head (lph lanes per head) and makes the same plan from them --
// totals, capacity checks before any write, pages bump-allocated in head order
// -- so no workgroup waits for another; then it compacts its own positions
// into the head's pages (new pages are numbered arithmetically from the plan,
// so the block-table entries written here are not read back) and writes the
// column counts of the row blocks whose band starts inside them: the count of
// row block r is the number of admitted positions below p = 64 r - W + 1,
// i.e. the inclusive count at virtual index p - 1 - base, the first of a
// step.  The global lengths and the bump pointer are left to stage 1 (every
// workgroup here reads the lengths from before the chunk).
//
// Bound by latency: the launch waits on memory about three times (flags and
// lengths, the head's last page id, K/V rows).  64 positions per workgroup
// give 512 workgroups for a 4096-token chunk of 8 heads, each copying its
// ~13 rows in one batch of loads.  Launched back to back, W 1024, a later
// 4096-token chunk: 8 heads 8.0 us (512 positions and one copy in flight per
// thread took 11.4, with the counts added into LDS by every thread), 32 heads
// 16.5 (29.4), 64 heads 27.4 (62.9); 64 tokens, W 64: 8 heads 4.8 (5.8), 64
// heads 4.9 (5.9).  span grows with heads x positions and lph falls with the
// heads (both in wgkv_chunk_cache_update).
__global__ __launch_bounds__(kThreads) void chunk_admit_kernel(ChunkArgs a) {
  __shared__ int s_tot[kMaxHeads];    // admitted positions of each head
  __shared__ int s_wave[kWaves];
  __shared__ int s_first, s_fail, s_total_pages;
  __shared__ int s_src[kBlk];         // row of the step's source
  __shared__ int64_t s_dst[kBlk];     // pool row
  const int h = blockIdx.y, tile = blockIdx.x;
  const int t = threadIdx.x;
  const int lane = t & 63, wid = t >> 6;
  const int nr = vring(a);
  const int n_adm = vlen(a) - a.W;  // admission range [0, n_adm) of the virtual sequence
  const int lb = a.W / a.page;
  const int v0 = tile * a.span * kBlk;
  const int32_t* lens = a.global_lengths + a.layer * a.H;
  int32_t* bt = a.block_table + ((int64_t)a.layer * a.H + h) * a.max_pages + lb;
  const uint8_t* ring_flags = a.local_is_global + ((int64_t)a.layer * a.H + h) * a.W;

  const int nf = *a.next_free;
  const int gl0 = lens[h];
  const int gl_t = lane < a.H ? lens[lane] : 0;
  const int open_page = gl0 % a.page ? bt[gl0 / a.page] : 0;  // the head's last page, partly filled

  // ---- admitted counts of every head, and of this head before v0 ----------
  const int lph = a.lph, sub = t & (lph - 1);
  for (int h0 = 0; h0 < a.H; h0 += kThreads / lph) {
    const int hh = h0 + t / lph;
    const int c = group_sum_int(hh < a.H ? vcount(a, hh, n_adm, sub, lph) : 0, lph);
    if (sub == 0 && hh < a.H) s_tot[hh] = c;
  }
  const int pre = wave_sum_int(v0 > 0 ? vcount(a, h, min(v0, n_adm), t, kThreads) : 0);
  if (lane == 0) s_wave[wid] = pre;
  __syncthreads();

  // ---- the plan (identical in every workgroup) ----------------------------
  if (wid == 0) {
    int carry = 0, bad = 0;
    for (int h0 = 0; h0 < a.H; h0 += 64) {
      const int hh = h0 + lane;
      int pages = 0;
      if (hh < a.H) {
        const int n = s_tot[hh];
        const int gl = h0 == 0 ? gl_t : lens[hh];
        pages = (gl + n + a.page - 1) / a.page - (gl + a.page - 1) / a.page;
        if (n > 0 && (a.W + gl + n > a.max_tokens_per_head || lb + (gl + n + a.page - 1) / a.page > a.max_pages)) bad = 1;
      }
      const int incl = wave_incl_scan(pages, lane);
      if (hh == h) s_first = carry + incl - pages;
      carry += __builtin_amdgcn_readlane(incl, 63);
    }
    bad = __builtin_amdgcn_ballot_w64(bad != 0) != 0;
    if (lane == 0) {
      s_total_pages = carry;
      s_fail = bad || (int64_t)nf + carry > a.total_pages;
    }
  }
  __syncthreads();
  const bool fail = s_fail != 0;
  int32_t* cc = a.column_count + (int64_t)h * a.rchunk;
  if (tile == 0) {
    // rows whose band starts at position 0 see no admitted column; on a
    // failure no row does (the chunk then attends to its band only)
    for (int i = t; i < a.rchunk; i += kThreads)
      if (fail || (a.r0 + i) * kBlk - a.W + 1 <= 0) cc[i] = 0;
    if (fail && h == 0 && t == 0) {
      *a.status = WGKV_ERR_CAPACITY;
      *a.abort_flag = 1;
    }
  }
  if (fail) return;  // tile 0 of each head has zeroed its column counts

  // ---- this workgroup's steps: stable compaction and column counts ---------
  const int first_new = (gl0 + a.page - 1) / a.page;  // index of the head's first new page
  const int page0 = nf + s_first;                       // its page id
  if (tile == 0) {
    const int n_h = s_tot[h];
    const int pages = (gl0 + n_h + a.page - 1) / a.page - first_new;
    for (int i = t; i < pages; i += kThreads) bt[first_new + i] = page0 + i;
    if (t == 0) {
      a.adm[h] = n_h;
      a.gl_before[h] = gl0;
      if (h == 0) {
        *a.next_free_after = nf + s_total_pages;
        *a.abort_flag = 0;
      }
    }
  }
  const int base = a.c0 > 0 ? a.c0 - a.W : 0;  // global position of virtual index 0
  const int64_t ring_base = ((int64_t)a.layer * a.H + h) * a.W;
  int before = gl0 + (s_wave[0] + s_wave[1]) + (s_wave[2] + s_wave[3]);
  for (int v = v0; v < min(n_adm, v0 + a.span * kBlk); v += kBlk) {
    // the step lies all in the ring or all in the chunk (W is a multiple of 64)
    const bool in_ring = v < nr;
    const uint8_t* fl = in_ring ? ring_flags + v : a.mask + (int64_t)h * a.m_sh + (v - nr);
    const uint64_t adm = __builtin_amdgcn_ballot_w64(v + lane < n_adm && fl[lane] != 0);
    if (wid == 0) {
      if (adm >> lane & 1) {
        const int o = __builtin_popcountll(adm & ((1ull << lane) - 1));
        const int j = before + o;  // logical index in the head's global cache
        const int pi = j / a.page;
        const int pg = pi < first_new ? open_page : page0 + (pi - first_new);
        s_src[o] = (in_ring ? v : v - nr) + lane;
        s_dst[o] = (int64_t)pg * a.page + (j - pi * a.page);
      }
      const int r = (base + v + a.W) / kBlk;  // the row block whose band starts at this step's second position
      if (lane == 0 && r >= a.r0 && r < a.r0 + a.rchunk) cc[r - a.r0] = before + (int)(adm & 1);
    }
    __syncthreads();
    const int n = __builtin_popcountll(adm);
    copy_rows2<kThreads>(in_ring ? a.pool_k + ring_base * a.D : a.key + (int64_t)h * a.kv_sh,
                         in_ring ? a.pool_v + ring_base * a.D : a.value + (int64_t)h * a.kv_sh,
                         in_ring ? (int64_t)a.D : a.kv_ss, n, a.D, [&](unsigned r) { return s_src[r]; },
                         [&](unsigned r) { return s_dst[r]; }, a.pool_k, a.pool_v);
    before += n;
    __syncthreads();
  }
}

// After the chunk's attention: ring slot i <- chunk position C - W + i.
// Grid (head, 64-slot group); a thread's rows are all requested before the
// first store (one at a time: 9.3 us for 8 heads of W 1024 with the pre-RoPE
// keys, median of a trace; 6.7 us).
__global__ __launch_bounds__(kThreads) void chunk_ring_kernel(ChunkArgs a) {
  if (*a.abort_flag) return;
  const int h = blockIdx.x;
  if (blockIdx.y == 0 && threadIdx.x == 0) {
    // stage 0's admissions become the head's global length (no kernel of
    // stage 0 could, since all of them read the length from before)
    a.global_lengths[a.layer * a.H + h] = a.gl_before[h] + a.adm[h];
    if (h == 0) *a.next_free = *a.next_free_after;
  }
  const int n_loc = min(a.W, a.c0 + a.C);
  const int first = a.C - n_loc;  // chunk row of slot 0
  const int i0 = blockIdx.y * kBlk, i1 = min(n_loc, i0 + kBlk);
  if (i0 >= i1) return;
  const int64_t ring_base = ((int64_t)a.layer * a.H + h) * a.W;
  copy_rows2<kThreads>(a.key + (int64_t)h * a.kv_sh, a.value + (int64_t)h * a.kv_sh, a.kv_ss, i1 - i0, a.D,
                       [&](unsigned r) { return first + i0 + (int)r; }, [&](unsigned r) { return ring_base + i0 + r; },
                       a.pool_k, a.pool_v);
  if (a.pre_key && a.local_pre_key)
    copy_rows1<kThreads>(a.pre_key + (int64_t)h * a.pk_sh, a.pk_ss, i1 - i0, a.D,
                         [&](unsigned r) { return first + i0 + (int)r; }, [&](unsigned r) { return ring_base + i0 + r; },
                         a.local_pre_key);
  for (int i = i0 + threadIdx.x; i < i1; i += kThreads)
    a.local_is_global[ring_base + i] = a.mask[(int64_t)h * a.m_sh + first + i] ? 1 : 0;
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

extern "C" size_t wgkv_chunk_admit_workspace_bytes(int32_t num_kv_heads, int32_t chunk_len, int32_t local_window) {
  (void)chunk_len;
  (void)local_window;
  return (2 * (size_t)(num_kv_heads > 0 ? num_kv_heads : 0) + 16) * sizeof(int32_t);
}

extern "C" int wgkv_chunk_cache_update(
    int32_t stage,
    const void* key, const void* value, int64_t kv_stride_h, int64_t kv_stride_s,
    const void* pre_key, int64_t pk_stride_h, int64_t pk_stride_s,
    const uint8_t* g_mask, int64_t gm_stride_h,
    int32_t layer, int32_t num_layers, int32_t num_kv_heads, int32_t chunk_start, int32_t chunk_len, int32_t head_dim,
    int32_t local_window, int32_t page_size, int32_t max_tokens_per_head, int64_t total_pages,
    void* pool_k, void* pool_v, int32_t* block_table, int32_t max_pages_per_head,
    int32_t* global_lengths, uint8_t* local_is_global, void* local_pre_key,
    int32_t* next_free_block, int32_t* status, int32_t* column_count,
    void* workspace, size_t workspace_bytes, void* stream) {
  if (stage != 0 && stage != 1) return WGKV_ERR_ARG;
  if (!key || !value || !g_mask || !pool_k || !pool_v || !block_table || !global_lengths || !local_is_global ||
      !next_free_block || !status)
    return WGKV_ERR_ARG;
  if (stage == 0 && !column_count) return WGKV_ERR_ARG;
  if (num_kv_heads <= 0 || num_kv_heads > 1024 || layer < 0 || layer >= num_layers) return WGKV_ERR_ARG;
  if (chunk_start < 0 || chunk_len <= 0 || local_window <= 0 || page_size <= 0) return WGKV_ERR_ARG;
  if (local_window % kBlk || chunk_start % kBlk || local_window % page_size) return WGKV_ERR_ARG;
  if (chunk_start > 0 && (chunk_len < local_window || chunk_start < local_window)) return WGKV_ERR_ARG;
  if (head_dim % 8 || head_dim <= 0) return WGKV_ERR_UNSUPPORTED;
  if (!aligned16(key) || !aligned16(value) || !aligned16(pool_k) || !aligned16(pool_v)) return WGKV_ERR_UNSUPPORTED;
  if ((kv_stride_h | kv_stride_s) & 7) return WGKV_ERR_UNSUPPORTED;
  if (pre_key && (!aligned16(pre_key) || ((pk_stride_h | pk_stride_s) & 7))) return WGKV_ERR_UNSUPPORTED;
  if (!workspace || workspace_bytes < wgkv_chunk_admit_workspace_bytes(num_kv_heads, chunk_len, local_window))
    return WGKV_ERR_WORKSPACE;
  ChunkArgs a = {};
  a.key = (const uint16_t*)key;
  a.value = (const uint16_t*)value;
  a.kv_sh = kv_stride_h;
  a.kv_ss = kv_stride_s;
  a.pre_key = (const uint16_t*)pre_key;
  a.pk_sh = pk_stride_h;
  a.pk_ss = pk_stride_s;
  a.mask = g_mask;
  a.m_sh = gm_stride_h;
  a.layer = layer;
  a.H = num_kv_heads;
  a.C = chunk_len;
  a.D = head_dim;
  a.W = local_window;
  a.page = page_size;
  a.max_tokens_per_head = max_tokens_per_head;
  a.c0 = chunk_start;
  a.total_pages = total_pages;
  a.pool_k = (uint16_t*)pool_k;
  a.pool_v = (uint16_t*)pool_v;
  a.block_table = block_table;
  a.max_pages = max_pages_per_head;
  a.global_lengths = global_lengths;
  a.local_is_global = local_is_global;
  a.local_pre_key = (uint16_t*)local_pre_key;
  a.next_free = next_free_block;
  a.status = status;
  a.column_count = column_count;
  a.r0 = chunk_start / kBlk;
  a.rchunk = (chunk_len + kBlk - 1) / kBlk;
  // 64-position steps of the admission range, and how many a workgroup takes:
  // one while the grid is small; more, up to kMaxSpan, where the counting that
  // every workgroup repeats would outweigh its own steps
  const int steps = (max(1, vlen(a) - local_window) + kBlk - 1) / kBlk;
  a.span = min(kMaxSpan, max(1, (int)((int64_t)steps * num_kv_heads / 1024)));
  // Lanes per head for the counting: the number that takes the fewest memory
  // round trips (count_flags has four 16-flag loads per lane in flight, and a
  // pass counts kThreads / lph heads).  A wave for every head took 17.3 us
  // instead of 4.9 for 64 heads of 64 tokens, 35.5 instead of 10.4 for 1000,
  // 24.5 instead of 16.5 for 32 heads of 4096.
  const int gr = vring(a) / 16, gc = (max(0, vlen(a) - local_window - vring(a)) + 15) / 16;
  int64_t best = INT64_MAX;
  for (int l = 64; l >= 1; l /= 4) {
    const int64_t trips = (int64_t)((num_kv_heads * l + kThreads - 1) / kThreads) * ((gr + 4 * l - 1) / (4 * l) + (gc + 4 * l - 1) / (4 * l));
    if (trips < best) {
      best = trips;
      a.lph = l;
    }
  }
  int32_t* ws = (int32_t*)workspace;
  a.adm = ws;
  a.gl_before = ws + num_kv_heads;
  a.next_free_after = ws + 2 * (size_t)num_kv_heads;
  a.abort_flag = a.next_free_after + 1;
  hipStream_t st = (hipStream_t)stream;
  if (stage == 0) {
    hipLaunchKernelGGL(chunk_admit_kernel, dim3((steps + a.span - 1) / a.span, num_kv_heads), dim3(kThreads), 0, st, a);
  } else {
    const int groups = (min(local_window, chunk_start + chunk_len) + kBlk - 1) / kBlk;
    hipLaunchKernelGGL(chunk_ring_kernel, dim3(num_kv_heads, groups), dim3(kThreads), 0, st, a);
  }
  return hipGetLastError() == hipSuccess ? WGKV_OK : WGKV_ERR_HIP;
}
