// Shared helpers of the gfx950 library: status codes, the thread-local error
// string behind dax_hip_last_error(), and wave64 primitives (DPP scans,
// ballots) used by the scan, compaction and marching-cubes kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include "../../include/dax_hip.h"

namespace daxhip {

void set_error(const char* fmt, ...);
int check_hip(hipError_t e, const char* what);

// Temporaries of the library's own launches: stream-ordered allocations from
// a per-device memory pool that keeps its memory between calls (no device
// synchronisation on free, no fresh mapping per call).
int temp_alloc(void** p, size_t bytes, hipStream_t s);
void temp_free(void* p, hipStream_t s);

// RAII holder of one temporary, released in stream order.
struct TempBuf {
  void* p = nullptr;
  hipStream_t s = nullptr;
  explicit TempBuf(hipStream_t stream) : s(stream) {}
  ~TempBuf() { temp_free(p, s); }
  TempBuf(const TempBuf&) = delete;
  TempBuf& operator=(const TempBuf&) = delete;
  int alloc(size_t bytes) { return temp_alloc(&p, bytes, s); }
  void release() {  // early, in stream order as well
    temp_free(p, s);
    p = nullptr;
  }
};

// Eight 64-bit words of pinned host memory that kernels write results into, so
// that a size reaches the host with the end of the kernel that has it: no
// copy launch and no staging buffer between.  From a fixed table of slots
// (one page, kept until the process ends), held by one call at a time; `p` is
// null when every slot is taken or there is no pinned memory, and the caller
// then copies.  A slot goes to another call only when the kernels of its
// holder's stream have ended: the holder waits for them with wait(), or (where
// it returns early with an error) its destructor does; a slot whose stream
// cannot be waited for is not given out again.
struct HostSlot {
  int64_t* p = nullptr;
  explicit HostSlot(hipStream_t stream);
  ~HostSlot();
  HostSlot(const HostSlot&) = delete;
  HostSlot& operator=(const HostSlot&) = delete;
  hipError_t wait();

 private:
  hipStream_t s_;
  int index_ = -1;
  bool waited_ = false;
};

#define DAXHIP_CHECK(expr)                                  \
  do {                                                      \
    hipError_t _e = (expr);                                 \
    if (_e != hipSuccess) return ::daxhip::check_hip(_e, #expr); \
  } while (0)

#define DAXHIP_LAUNCH_CHECK(what)                            \
  do {                                                      \
    hipError_t _e = hipGetLastError();                      \
    if (_e != hipSuccess) return ::daxhip::check_hip(_e, what); \
  } while (0)

// Inclusive prefix sum over the 64 lanes of a wavefront with DPP row shifts
// and the GFX9 row broadcasts (row_shr:1/2/4/8, row_bcast:15, row_bcast:31).
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);
  return v;
}

// Value of lane 63 broadcast to the whole wave.
__device__ __forceinline__ uint32_t wave_last(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t v) { return wave_last(wave_incl_scan(v)); }

// Exclusive scan of one value per thread over the block (thread order);
// returns the thread's offset and the block total.
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t& total, uint32_t* s_w) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nwv = blockDim.x >> 6;
  const uint32_t inc = wave_incl_scan(v);
  if (lane == 63) s_w[wv] = inc;
  __syncthreads();
  uint32_t off = 0, tot = 0;
  for (int q = 0; q < nwv; ++q) {
    if (q < wv) off += s_w[q];
    tot += s_w[q];
  }
  __syncthreads();
  total = tot;
  return off + inc - v;
}

// Orders the LDS accesses of a wave's lanes among themselves (a wave's LDS
// operations execute in order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Inclusive prefix maximum over the lanes of a wave (wave_incl_scan's steps).
__device__ __forceinline__ uint32_t wave_incl_max(uint32_t v) {
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));
  return v;
}

// Position of the k-th set bit of m (k < popcount(m)): the half of m that
// holds it, then halving steps on 32 bits.
__device__ __forceinline__ int select_bit(uint64_t m, int k) {
  const uint32_t lo = (uint32_t)m;
  const int nlo = __popc(lo);
  const bool up = k >= nlo;
  uint32_t x = up ? (uint32_t)(m >> 32) : lo;
  int r = up ? k - nlo : k, pos = up ? 32 : 0;
#pragma unroll
  for (int w = 16; w > 0; w >>= 1) {
    const int c = __popc(x & ((1u << w) - 1u));
    const bool hi = r >= c;
    r = hi ? r - c : r;
    x = hi ? x >> w : x;
    pos += hi ? w : 0;
  }
  return pos;
}

// The thread's kScanChunk values [i0, i0 + kScanChunk) of n (zeros past the
// end) and their exclusive prefixes back, in 16-byte pieces where the array is
// aligned: a block that scans many values is bound by its round trips, and
// with single accesses at a stride a round of 8 values a thread took 5 us.
constexpr int kScanChunk = 16;
using u32x4 = uint32_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void load_chunk(const uint32_t* __restrict__ v, int64_t i0, int64_t n,
                                           u32x4 (&x)[kScanChunk / 4]) {
  const bool whole = i0 + kScanChunk <= n && (reinterpret_cast<uintptr_t>(v) & 15u) == 0;
#pragma unroll
  for (int q = 0; q < kScanChunk / 4; ++q) {
    if (whole) {
      x[q] = *reinterpret_cast<const u32x4*>(v + i0 + 4 * q);
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t) x[q][t] = i0 + 4 * q + t < n ? v[i0 + 4 * q + t] : 0u;
    }
  }
}
__device__ __forceinline__ void store_prefixes(uint32_t* __restrict__ v, int64_t i0, int64_t n,
                                               u32x4 (&x)[kScanChunk / 4], uint32_t run) {
#pragma unroll
  for (int q = 0; q < kScanChunk; ++q) {
    const uint32_t t = x[q / 4][q % 4];
    x[q / 4][q % 4] = run;
    run += t;
  }
  const bool whole = i0 + kScanChunk <= n && (reinterpret_cast<uintptr_t>(v) & 15u) == 0;
#pragma unroll
  for (int q = 0; q < kScanChunk / 4; ++q) {
    if (whole) {
      *reinterpret_cast<u32x4*>(v + i0 + 4 * q) = x[q];
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (i0 + 4 * q + t < n) v[i0 + 4 * q + t] = x[q][t];
    }
  }
}

__host__ __device__ __forceinline__ int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

__host__ __device__ __forceinline__ size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

}  // namespace daxhip
