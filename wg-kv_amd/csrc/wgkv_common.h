// Shared device helpers for the write-gated dual-cache kernels (gfx950 only).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/wgkv.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4_t;

#define WGKV_DEVICE __device__ __forceinline__

// ---- bf16 <-> f32 ---------------------------------------------------------
// A bf16 value is the high half of an f32, so widening is a shift / mask.
WGKV_DEVICE float bf16lo(uint32_t w) { return __uint_as_float(w << 16); }
WGKV_DEVICE float bf16hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// Two f32 -> packed bf16 pair, round to nearest even (v_cvt_pk_bf16_f32).
WGKV_DEVICE uint32_t pack_bf16x2(float lo, float hi) {
  typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2_t;
  bf16x2_t r;
  r[0] = (__bf16)lo;
  r[1] = (__bf16)hi;
  return __builtin_bit_cast(uint32_t, r);
}

// Round-to-nearest-even f32 -> bf16 (NaN kept quiet).
WGKV_DEVICE uint16_t f32_to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

// f32 rounded to the nearest bf16 (ties to even) and widened back: one
// v_cvt_pk_bf16_f32 and a shift.
WGKV_DEVICE float round_to_bf16(float x) { return (float)(__bf16)x; }

// ---- DPP row (16-lane) reductions -----------------------------------------
// quad_perm(1,0,3,2), quad_perm(2,3,0,1), row_half_mirror, row_mirror: after
// the four steps every lane of a 16-lane row holds the row-wide result.
#define WGKV_DPP_QP_1032 0xB1
#define WGKV_DPP_QP_2301 0x4E
#define WGKV_DPP_ROW_MIRROR 0x140
#define WGKV_DPP_ROW_HALF_MIRROR 0x141

template <int CTRL>
WGKV_DEVICE float dpp_f32(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, false));
}

WGKV_DEVICE float row_max16(float x) {
  x = fmaxf(x, dpp_f32<WGKV_DPP_QP_1032>(x));
  x = fmaxf(x, dpp_f32<WGKV_DPP_QP_2301>(x));
  x = fmaxf(x, dpp_f32<WGKV_DPP_ROW_HALF_MIRROR>(x));
  x = fmaxf(x, dpp_f32<WGKV_DPP_ROW_MIRROR>(x));
  return x;
}

WGKV_DEVICE float row_sum16(float x) {
  x += dpp_f32<WGKV_DPP_QP_1032>(x);
  x += dpp_f32<WGKV_DPP_QP_2301>(x);
  x += dpp_f32<WGKV_DPP_ROW_HALF_MIRROR>(x);
  x += dpp_f32<WGKV_DPP_ROW_MIRROR>(x);
  return x;
}

// Wave-uniform max / sum over all 64 lanes.
WGKV_DEVICE float wave_max(float x) {
  x = row_max16(x);
  float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 0));
  float b = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 16));
  float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 32));
  float d = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 48));
  return fmaxf(fmaxf(a, b), fmaxf(c, d));
}

WGKV_DEVICE float wave_sum(float x) {
  x = row_sum16(x);
  float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 0));
  float b = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 16));
  float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 32));
  float d = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 48));
  return (a + b) + (c + d);
}

// Inclusive prefix sum over the 64 lanes of a wave.
WGKV_DEVICE int wave_incl_scan(int v, int lane) {
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int u = __shfl_up(v, off, 64);
    if (lane >= off) v += u;
  }
  return v;
}

// Sum of an int over an aligned group of n lanes, n one of 1, 4, 16, 64 and
// the same in the whole wave (every lane of the group gets the total).
WGKV_DEVICE int group_sum_int(int x, int n) {
  if (n >= 4) {
    x += __builtin_amdgcn_update_dpp(0, x, WGKV_DPP_QP_1032, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, WGKV_DPP_QP_2301, 0xf, 0xf, false);
  }
  if (n >= 16) {
    x += __builtin_amdgcn_update_dpp(0, x, WGKV_DPP_ROW_HALF_MIRROR, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, WGKV_DPP_ROW_MIRROR, 0xf, 0xf, false);
  }
  if (n == 64)
    x = (__builtin_amdgcn_readlane(x, 0) + __builtin_amdgcn_readlane(x, 16)) +
        (__builtin_amdgcn_readlane(x, 32) + __builtin_amdgcn_readlane(x, 48));
  return x;
}

// Sum of an int over all 64 lanes (every lane gets the total).
WGKV_DEVICE int wave_sum_int(int x) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
  return x;
}

WGKV_DEVICE float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Orders this wave's LDS writes before its later LDS reads of other lanes'
// data (LDS operations of one wave complete in issue order).
WGKV_DEVICE void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Block-wide exclusive scan of one int per thread (blockDim.x == 256): a
// wave prefix sum, then the four wave totals through LDS (two barriers).
WGKV_DEVICE int block_exclusive_scan_256(int v, int* s_tmp /* >= 4 ints */, int* total) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int incl = wave_incl_scan(v, lane);
  if (lane == 63) s_tmp[w] = incl;
  __syncthreads();
  const int t0 = s_tmp[0], t1 = s_tmp[1], t2 = s_tmp[2], t3 = s_tmp[3];
  const int before = (w > 0 ? t0 : 0) + (w > 1 ? t1 : 0) + (w > 2 ? t2 : 0);
  if (total) *total = (t0 + t1) + (t2 + t3);
  __syncthreads();
  return before + incl - v;
}

// This thread's share (t of n threads) of the nonzero flags in
// m[lo, hi): whole 16-byte groups as vectors, the ends -- rows of odd length
// start anywhere -- as bytes.
WGKV_DEVICE int count_flags(const uint8_t* m, int lo, int hi, int t, int n) {
  if (hi <= lo) return 0;
  const uint8_t* p = m + lo;
  const int head = min((int)((16 - ((uintptr_t)p & 15)) & 15), hi - lo);
  const int groups = (hi - lo - head) >> 4;
  const int tail = hi - lo - head - groups * 16;
  int c = 0;
  for (int i = t; i < head; i += n) c += p[i] != 0;
  for (int i = t; i < tail; i += n) c += m[hi - tail + i] != 0;
  const u32x4_t* v = (const u32x4_t*)(p + head);
  constexpr int U = 4;  // loads in flight
  for (int g0 = t; g0 < groups; g0 += n * U) {
    u32x4_t w[U];
#pragma unroll
    for (int u = 0; u < U; ++u) w[u] = v[min(g0 + u * n, groups - 1)];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      int k = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i)  // bit 7 of each nonzero byte
        k += __builtin_popcount((((w[u][i] & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w[u][i]) & 0x80808080u);
      c += g0 + u * n < groups ? k : 0;
    }
  }
  return c;
}

// Copies rows r < n of one K/V pair (source row src(r), pool row dst(r)) with
// the whole workgroup of kThreads, 16 bytes per thread and step.  Eight loads per thread
// are requested before the first store: one load and one store at a time
// waited for memory once per step (64 us of a 9001-token prompt's 76).
template <int kThreads, typename Src, typename Dst>
WGKV_DEVICE void copy_rows2(const uint16_t* ka, const uint16_t* va, int64_t ss, int n, int D, Src src, Dst dst,
                            uint16_t* pool_k, uint16_t* pool_v) {
  constexpr int U = 4;
  const unsigned chunks = D / 8;
  const unsigned total = n * chunks;
  for (unsigned e0 = threadIdx.x; e0 < total; e0 += kThreads * U) {
    u32x4_t k[U], v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const unsigned e = min(e0 + u * kThreads, total - 1);
      const unsigned r = e / chunks;
      const int64_t off = (int64_t)src(r) * ss + (e - r * chunks) * 8;
      k[u] = *(const u32x4_t*)(ka + off);
      v[u] = *(const u32x4_t*)(va + off);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const unsigned e = e0 + u * kThreads;
      if (e >= total) break;
      const unsigned r = e / chunks;
      const int64_t off = dst(r) * D + (e - r * chunks) * 8;
      *(u32x4_t*)(pool_k + off) = k[u];
      *(u32x4_t*)(pool_v + off) = v[u];
    }
  }
}

// The same for one array.
template <int kThreads, typename Src, typename Dst>
WGKV_DEVICE void copy_rows1(const uint16_t* a, int64_t ss, int n, int D, Src src, Dst dst, uint16_t* to) {
  constexpr int U = 4;
  const unsigned chunks = D / 8;
  const unsigned total = n * chunks;
  for (unsigned e0 = threadIdx.x; e0 < total; e0 += kThreads * U) {
    u32x4_t v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const unsigned e = min(e0 + u * kThreads, total - 1);
      const unsigned r = e / chunks;
      v[u] = *(const u32x4_t*)(a + (int64_t)src(r) * ss + (e - r * chunks) * 8);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const unsigned e = e0 + u * kThreads;
      if (e >= total) break;
      const unsigned r = e / chunks;
      *(u32x4_t*)(to + dst(r) * D + (e - r * chunks) * 8) = v[u];
    }
  }
}

// Compute units of the current device (256 where it cannot be asked).
inline int cu_count() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cached[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cached[dev] = n;
  }
  return cached[dev];
}

#define WGKV_HIP_CHECK(expr)                       \
  do {                                             \
    hipError_t _e = (expr);                        \
    if (_e != hipSuccess) return WGKV_ERR_HIP;     \
  } while (0)
