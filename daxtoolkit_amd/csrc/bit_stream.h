// Words of 64 bits along the rows of a grid, made from and turned into flat
// arrays: a predicate of every value of an array as one bit (classify_flat),
// and every bit as an int32 (store_words_i32).  A run of row words covers one
// contiguous run of the array, so both read and write it in aligned 16-byte
// pieces whatever the rows' extents and the array's alignment.
#pragma once

#include "mc_common.h"

namespace daxhip {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));

// Rows of nx values in wpr = ceil(nx / 64) words each, `total` values in all.
struct FlatRows {
  int32_t nx, wpr, total;
  mc::FastDiv div_wpr;
};

__device__ __forceinline__ int32_t first_value(const FlatRows& r, uint32_t w, uint32_t& q) {
  const uint32_t row = mc::fast_div(w, r.div_wpr);
  q = w - row * (uint32_t)r.wpr;
  return (int32_t)(row * (uint32_t)r.nx + 64u * q);
}

// OR of the 16 lanes' nibbles (4 bits, lane l of a row at bits 4l .. 4l+3)
// in lane 15 of every 16-lane row, in steps of 1, 2, 4 and 8 lanes.
__device__ __forceinline__ uint64_t row_nibbles(uint32_t nib, int lane) {
  const int sh = 4 * (lane & 15);
  uint32_t lo = sh < 32 ? nib << sh : 0u;
  uint32_t hi = sh >= 32 ? nib << (sh - 32) : 0u;
  lo |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)lo, 0x111, 0xf, 0xf, false);
  hi |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)hi, 0x111, 0xf, 0xf, false);
  lo |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)lo, 0x112, 0xf, 0xf, false);
  hi |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)hi, 0x112, 0xf, 0xf, false);
  lo |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)lo, 0x114, 0xf, 0xf, false);
  hi |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)hi, 0x114, 0xf, 0xf, false);
  lo |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)lo, 0x118, 0xf, 0xf, false);
  hi |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)hi, 0x118, 0xf, 0xf, false);
  return ((uint64_t)hi << 32) | lo;
}

// Row words [w0, w_end) (at most TW, a block of 256 threads) of pred(value):
// the values are read as a flat stream of aligned float4s, their bits go to
// LDS in stream order, and each thread cuts its row words out of two
// neighbouring stream words.  A lane per value of a row word instead leaves
// the lanes past a row's end idle and takes four times the load
// instructions: the inside-bits of 301 x 257 x 190 points took 35 us that way
// and take 12 (4.9 TB/s), of 256 volumes of 32..160 points an axis (0.9 GB)
// 645 us and 180 (5.1 TB/s).
template <int TW>
struct FlatLds {
  uint64_t w[TW + 4];  // stream words of at most 64 TW + 3 values, read one past the end
};
constexpr int kFlatLoads = 8;  // float4 loads in flight per thread

template <int TW, int LOADS, class Pred>
__device__ __forceinline__ void classify_flat(const FlatRows& rows, const float* __restrict__ f,
                                              uint64_t* __restrict__ bits, uint32_t w0,
                                              uint32_t w_end, FlatLds<TW>& sh, Pred pred) {
  const int tid = threadIdx.x, lane = tid & 63;
  uint32_t qa, qb;
  const int32_t p0 = first_value(rows, w0, qa);
  const int32_t pl = first_value(rows, w_end - 1, qb);
  const int32_t p1 = pl + min(64, rows.nx - (int32_t)(64u * qb));
  // stream position 0 is the 16-byte boundary at or below value p0
  const int32_t e0 = p0 - (int32_t)((reinterpret_cast<uintptr_t>(f + p0) >> 2) & 3u);
  const int32_t n4 = (p1 - e0 + 3) >> 2;
  for (int32_t b = 0; b < n4; b += LOADS * 256) {
    f32x4 v[LOADS];
#pragma unroll
    for (int u = 0; u < LOADS; ++u) {
      const int32_t i = b + u * 256 + tid;
      const int64_t e = (int64_t)e0 + 4 * (int64_t)i;
      v[u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      if (i < n4) {
        if (e >= 0 && e + 4 <= rows.total) {
          v[u] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(f + e));
        } else {  // the stream's first or last float4 crosses the array's ends
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (e + c >= 0 && e + c < rows.total) v[u][c] = f[e + c];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < LOADS; ++u) {
      const int32_t i = b + u * 256 + tid;
      const uint32_t nib = (uint32_t)pred(v[u].x) | ((uint32_t)pred(v[u].y) << 1) |
                           ((uint32_t)pred(v[u].z) << 2) | ((uint32_t)pred(v[u].w) << 3);
      const uint64_t word = row_nibbles(nib, lane);
      // the last stream word may be partly past n4: its bits are cut off below
      if ((lane & 15) == 15 && (i & ~15) < n4) sh.w[i >> 4] = word;
    }
  }
  __syncthreads();
  for (uint32_t w = w0 + (uint32_t)tid; w < w_end; w += 256u) {
    uint32_t q;
    const uint32_t s = (uint32_t)(first_value(rows, w, q) - e0);
    const uint64_t lo = sh.w[s >> 6], hi = sh.w[(s >> 6) + 1];
    const int r = (int)(s & 63u);
    const uint64_t m = r ? (lo >> r) | (hi << (64 - r)) : lo;
    bits[w] = m & mc::low_mask(rows.nx - (int)(64u * q));
  }
}

// The bits of row words [w0, w_end), s_w[0 .. w_end - w0) in LDS, as int32 0/1
// at their places in `out`: 16-byte non-temporal stores between scalar ends
// (all threads of a block).
__device__ __forceinline__ void store_words_i32(const FlatRows& rows, mc::FastDiv div_nx,
                                                const uint64_t* __restrict__ s_w, uint32_t w0,
                                                uint32_t w_end, int32_t* __restrict__ out) {
  uint32_t qa, qb;
  const int32_t p0 = first_value(rows, w0, qa);
  const int32_t pl = first_value(rows, w_end - 1, qb);
  const int32_t p1 = pl + min(64, rows.nx - (int32_t)(64u * qb));
  const int32_t e0 = p0 - (int32_t)((reinterpret_cast<uintptr_t>(out + p0) >> 2) & 3u);
  auto bit = [&](int32_t e) -> int32_t {
    const uint32_t row = mc::fast_div((uint32_t)e, div_nx), x = (uint32_t)e - row * (uint32_t)rows.nx;
    return (int32_t)((s_w[row * (uint32_t)rows.wpr + (x >> 6) - w0] >> (x & 63u)) & 1u);
  };
  const int32_t n4 = (int32_t)(((int64_t)p1 - e0 + 3) >> 2);
  for (int32_t i = (int32_t)threadIdx.x; i < n4; i += (int32_t)blockDim.x) {
    const int64_t e = (int64_t)e0 + 4 * (int64_t)i;
    if (e < p0 || e + 4 > p1) {
      for (int c = 0; c < 4; ++c)
        if (e + c >= p0 && e + c < p1) out[e + c] = bit((int32_t)(e + c));
      continue;
    }
    const uint32_t row = mc::fast_div((uint32_t)e, div_nx);
    const uint32_t x = (uint32_t)e - row * (uint32_t)rows.nx;
    i32x4 v;
    if (x + 4u <= (uint32_t)rows.nx) {
      const uint32_t li = row * (uint32_t)rows.wpr + (x >> 6) - w0, s = x & 63u;
      uint32_t b = (uint32_t)(s_w[li] >> s);
      if (s > 60u) b |= (uint32_t)(s_w[li + 1] << (64u - s));
      v = i32x4{(int32_t)(b & 1u), (int32_t)((b >> 1) & 1u), (int32_t)((b >> 2) & 1u),
                (int32_t)((b >> 3) & 1u)};
    } else {  // across a row's end
      v = i32x4{bit((int32_t)e), bit((int32_t)e + 1), bit((int32_t)e + 2), bit((int32_t)e + 3)};
    }
    __builtin_nontemporal_store(v, reinterpret_cast<i32x4*>(out + e));
  }
}

}  // namespace daxhip
