// Device bodies of the marching-cubes kernels, shared by the single-volume
// launches (mc_forward.hip) and the batched launches (mc_batched.hip).
//
//   classify   : field -> inside-bits                         (one pass over f)
//   count/scan : per-word edge and triangle counts, prefixes within count
//                tiles and blocks, one block scanning the blocks' sums
//   generate   : per generate tile, maps of the tile's output vertices and
//                triangles built in LDS, then one thread per vertex and per
//                triangle with coalesced writes
#pragma once

#include "bit_stream.h"
#include "mc_common.h"

namespace daxhip {
namespace mc {

// Case table in constant memory (one copy per translation unit).
static __constant__ uint64_t c_case_table[256] = DAX_HIP_MC_CASE_TABLE_INIT;

// ---------------------------------------------------------------------------
// Incremental word positions (32-bit arithmetic, one division per start).
struct WordIter {
  int q, j, k;
  __device__ __forceinline__ void init(const VolGeom& g, int lw) {
    const uint32_t row = fast_div((uint32_t)lw, g.div_wpr);
    const uint32_t kk = fast_div(row, g.div_ny);
    q = lw - (int)row * g.wpr;
    j = (int)(row - kk * (uint32_t)g.ny);
    k = (int)kk;
  }
  __device__ __forceinline__ void next(const VolGeom& g) {
    if (++q == g.wpr) {
      q = 0;
      if (++j == g.ny) {
        j = 0;
        ++k;
      }
    }
  }
  __device__ __forceinline__ WordPos pos(const VolGeom& g) const {
    WordPos p;
    p.q = q;
    p.j = j;
    p.k = k;
    p.has_y = j + 1 < g.ny;
    p.has_z = k + 1 < g.nz;
    const bool has_cells = g.nx > 1 && g.ny > 1 && g.nz > 1;
    const int x0 = q * 64;
    p.pmask = has_cells ? low_mask(g.nx - x0) : 0ull;
    p.xmask = has_cells ? low_mask(g.nx - 1 - x0) : 0ull;
    return p;
  }
};

// ---------------------------------------------------------------------------
// classify, one float per lane (rows of a multiple of 64 points): a wave
// builds UNROLL consecutive words.
template <int UNROLL>
__device__ __forceinline__ void classify_words(const VolGeom& g, const float* __restrict__ f,
                                               uint64_t* __restrict__ bits, int64_t w0,
                                               int64_t w_end) {
  const int lane = __lane_id();
  float v[UNROLL];
  bool ok[UNROLL];
#pragma unroll
  for (int u = 0; u < UNROLL; ++u) {
    const int64_t w = w0 + u;
    ok[u] = w < w_end;
    v[u] = ok[u] ? __builtin_nontemporal_load(f + w * 64 + lane) : 0.0f;
  }
  uint64_t mine = 0;
#pragma unroll
  for (int u = 0; u < UNROLL; ++u) {
    const uint64_t b = __ballot(ok[u] && v[u] > g.iso);
    if (lane == u) mine = b;
  }
  if (lane < UNROLL && w0 + lane < w_end) bits[w0 + lane] = mine;
}

// The volume's points as rows of a flat array (bit_stream.h).
__device__ __forceinline__ FlatRows flat_rows(const VolGeom& g) {
  return FlatRows{g.nx, g.wpr, g.nx * g.ny * g.nz, g.div_wpr};
}

// classify, float4 per lane (rows of a multiple of 64 points): a wave reads
// UNROLL chunks of 256 consecutive points; lane l holds points 4l..4l+3 of a
// chunk, and a DPP OR-scan over each 16-lane row assembles the chunk's four
// 64-bit words.
template <int UNROLL>
__device__ __forceinline__ void classify_chunks_v4(const VolGeom& g, const float* __restrict__ f,
                                                   uint64_t* __restrict__ bits, int64_t c0,
                                                   int64_t nwords) {
  const int lane = __lane_id();
  const f32x4* f4 = reinterpret_cast<const f32x4*>(f);
  f32x4 v[UNROLL];
  bool ok[UNROLL];
#pragma unroll
  for (int u = 0; u < UNROLL; ++u) {
    const int64_t c = c0 + u;
    ok[u] = (4 * c + (lane >> 4)) < nwords;
    v[u] = ok[u] ? __builtin_nontemporal_load(f4 + c * 64 + lane) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }
#pragma unroll
  for (int u = 0; u < UNROLL; ++u) {
    const float iso = g.iso;
    const uint32_t nib = (uint32_t)(v[u].x > iso) | ((uint32_t)(v[u].y > iso) << 1) |
                         ((uint32_t)(v[u].z > iso) << 2) | ((uint32_t)(v[u].w > iso) << 3);
    const uint64_t word = row_nibbles(nib, lane);
    if ((lane & 15) == 15 && ok[u]) bits[4 * (c0 + u) + (lane >> 4)] = word;
  }
}

// ---------------------------------------------------------------------------
// count/scan: every word's vertices and triangles, prefixes within tiles of
// kCountTile words, the tiles' within count blocks, and one block scanning the
// blocks' sums.
// Active edges (vertices) and triangles of one row word from its eight
// neighbour words (A = the word, 1 = the next word along x, B = +y row,
// C = +z plane, D = +y+z).
__device__ __forceinline__ void word_counts_regs(const VolGeom& g, const WordPos& p, uint64_t A,
                                                 uint64_t A1, uint64_t B, uint64_t B1, uint64_t C,
                                                 uint64_t C1, uint64_t D, uint64_t D1,
                                                 uint32_t& nv, uint32_t& nt) {
  uint64_t fx, fy, fz;
  edge_flags(p, A, A1, B, C, fx, fy, fz);
  nv = (uint32_t)(popc(fx) + popc(fy) + popc(fz));
  CellPlanes cp;
  cell_planes(p, A, A1, B, B1, C, C1, D, D1, cp);
  nt = cp.active ? word_triangles(cp) : 0u;
}

// Two count tiles of kCountTile row words, one wave: lane l counts the four
// consecutive words 2*kCountTile*pair + 4l .. +3 (lanes 0-31 the first
// tile, 32-63 the second), reusing each loaded word as its predecessor's +x
// neighbour, and writes each word's exclusive prefix within its tile
// (v | t << 16).  Returns the two tiles' sums (v | t << 32, wave-uniform).
__device__ __forceinline__ void count_tile_pair(const VolGeom& g, const uint64_t* __restrict__ b,
                                                uint32_t* __restrict__ lpre, int64_t pair,
                                                int64_t n_ctiles, unsigned long long& sum0,
                                                unsigned long long& sum1) {
  static_assert(kCountTile == 128, "32 lanes of four words per count tile");
  const int lane = __lane_id();
  const int64_t plane = (int64_t)g.wpr * g.ny;
  const int wpr = g.wpr;
  const int64_t w0 = pair * (2 * kCountTile) + 4 * lane;
  uint64_t A[5], B[5], C[5], D[5];
#pragma unroll
  for (int i = 0; i < 5; ++i) {
    const int64_t w = w0 + i;
    A[i] = w < g.nwords ? b[w] : 0ull;
    B[i] = w + wpr < g.nwords ? b[w + wpr] : 0ull;
    C[i] = w + plane < g.nwords ? b[w + plane] : 0ull;
    D[i] = w + plane + wpr < g.nwords ? b[w + plane + wpr] : 0ull;
  }
  uint32_t nv[4] = {0u, 0u, 0u, 0u}, nt[4] = {0u, 0u, 0u, 0u};
  if (w0 < g.nwords) {
    WordIter wi;
    wi.init(g, (int)w0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (w0 + i < g.nwords) {
        const WordPos p = wi.pos(g);
        const bool nx1 = p.q + 1 < wpr;
        word_counts_regs(g, p, A[i], nx1 ? A[i + 1] : 0ull, B[i], nx1 ? B[i + 1] : 0ull, C[i],
                         nx1 ? C[i + 1] : 0ull, D[i], nx1 ? D[i + 1] : 0ull, nv[i], nt[i]);
        wi.next(g);
      }
    }
  }
  const uint32_t sv = nv[0] + nv[1] + nv[2] + nv[3], st = nt[0] + nt[1] + nt[2] + nt[3];
  uint32_t iv = wave_incl_scan(sv), it = wave_incl_scan(st);
  const uint32_t hv = (uint32_t)__builtin_amdgcn_readlane((int)iv, 31);
  const uint32_t ht = (uint32_t)__builtin_amdgcn_readlane((int)it, 31);
  const uint32_t ev = (uint32_t)__builtin_amdgcn_readlane((int)iv, 63);
  const uint32_t et = (uint32_t)__builtin_amdgcn_readlane((int)it, 63);
  sum0 = (unsigned long long)hv | ((unsigned long long)ht << 32);
  sum1 = (unsigned long long)(ev - hv) | ((unsigned long long)(et - ht) << 32);
  if (lane >= 32) {  // the second tile's scan starts at lane 32
    iv -= hv;
    it -= ht;
  }
  const int64_t tile = pair * 2 + (lane >> 5);
  if (tile < n_ctiles) {
    uint32_t rv = iv - sv, rt = it - st;
    uint32_t out[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      out[i] = rv | (rt << 16);
      rv += nv[i];
      rt += nt[i];
    }
    *reinterpret_cast<uint4*>(lpre + w0) = make_uint4(out[0], out[1], out[2], out[3]);
  }
}

// Blocks are dispatched round-robin over the 8 XCDs; give each XCD a
// contiguous range of tiles so neighbouring tiles share its L2.
__device__ __forceinline__ int64_t xcd_tile(int64_t b, int64_t n) {
  const int64_t per = n / 8, rem = n % 8;
  const int64_t x = b % 8, i = b / 8;
  return x * per + (x < rem ? x : rem) + i;
}

// The same within groups of 8 * kXcdRun tiles, so that no XCD is left with a
// heavier part of the whole range.
constexpr int64_t kXcdRun = 32;
__device__ __forceinline__ int64_t xcd_tile_runs(int64_t b, int64_t n) {
  const int64_t g0 = b / (8 * kXcdRun) * (8 * kXcdRun);
  return g0 + xcd_tile(b - g0, min(8 * kXcdRun, n - g0));
}

// ---------------------------------------------------------------------------
// generate
struct OutPtrs {
  float* vertices;
  float* normals;
  int32_t* conn;
  uint32_t* edges;
  int32_t* interp_first;
  int32_t* interp_second;
  float* interp_weight;
};

// Point-field sources of the forward: a float32 field in memory, or the
// signed plane distance of a slice computed from the point's coordinates.
// src(x, y, z, p) is the value at point (x, y, z) of flat index p (a volume
// holds fewer than 2^31 points, so 32-bit index arithmetic is exact).
struct FieldArray {
  const float* __restrict__ f;
  __device__ __forceinline__ float operator()(int, int, int, int32_t p) const { return f[p]; }
};

// The field SliceCount / SliceGenerate classify and interpolate
// (dax/worklet/Slice.h:44-57,104-120): dot(normal, c - origin) at the point
// coordinates c = grid origin + spacing * ijk (dax/cont/UniformGrid.h:82-89),
// the dot product summed from component 0 (dax/Types.h:611-621), against
// the isovalue dot(normal, origin).
struct FieldPlane {
  float o[3], s[3];  // grid origin and spacing
  float po[3], pn[3];  // plane origin and normal
  __device__ __forceinline__ float operator()(int x, int y, int z, int32_t) const {
    const int c[3] = {x, y, z};
    float r = 0.0f;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const float t = pn[d] * ((o[d] + s[d] * (float)c[d]) - po[d]);
      r = d == 0 ? t : r + t;
    }
    return r;
  }
};

// Central-difference gradient at (x,y,z): interior (f(p+e)-f(p-e))/(2h),
// first plane (f(p+e)-f(p))/h, last plane (f(p)-f(p-e))/h, and 0 along an
// axis with a single point.  Split into the loads (branch-free, so they all
// issue at once) and the arithmetic, so callers can overlap other work with
// the loads' latency.
template <class Src>
__device__ __forceinline__ void gradient_loads(const VolGeom& g, const Src& f, int x, int y, int z,
                                               float lo_v[3], float hi_v[3]) {
  const int32_t sy = g.nx, sz = g.nx * g.ny;
  const int32_t p = x + sy * y + sz * z;
  const int c[3] = {x, y, z};
  const int n[3] = {g.nx, g.ny, g.nz};
  const int32_t st[3] = {1, sy, sz};
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const int dl = c[d] > 0 ? 1 : 0, dh = c[d] < n[d] - 1 ? 1 : 0;
    lo_v[d] = f(x - (d == 0) * dl, y - (d == 1) * dl, z - (d == 2) * dl, p - dl * st[d]);
    hi_v[d] = f(x + (d == 0) * dh, y + (d == 1) * dh, z + (d == 2) * dh, p + dh * st[d]);
  }
}

__device__ __forceinline__ void gradient_finish(const VolGeom& g, int x, int y, int z,
                                                const float lo_v[3], const float hi_v[3],
                                                float out[3]) {
  const int c[3] = {x, y, z};
  const int n[3] = {g.nx, g.ny, g.nz};
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const bool wide = c[d] > 0 && c[d] < n[d] - 1;
    const float h = g.spacing[d];
    const float diff = hi_v[d] - lo_v[d];
    if (n[d] < 2)
      out[d] = 0.0f;
    else if ((g.pow2_h >> d) & 1u)  // exact: the same value as the division
      out[d] = diff * (wide ? 0.5f * g.rcp_h[d] : g.rcp_h[d]);
    else
      out[d] = diff / (wide ? 2.0f * h : h);
  }
}

template <class Src>
__device__ __forceinline__ void point_gradient(const VolGeom& g, const Src& f, int x, int y,
                                               int z, float out[3]) {
  float lo_v[3], hi_v[3];
  gradient_loads(g, f, x, y, z, lo_v, hi_v);
  gradient_finish(g, x, y, z, lo_v, hi_v, out);
}

// Field values of one interpolated point on the edge with lower endpoint
// (x,y,z) along axis: the end values and, with normals, the central-
// difference neighbours of both ends.
struct PointLoads {
  float fa, fb;
  float alo[3], ahi[3], blo[3], bhi[3];
};

template <class Src>
__device__ __forceinline__ void point_loads(const VolGeom& g, const Src& f, int x, int y, int z,
                                            int axis, bool normals, PointLoads& L, int32_t& pa,
                                            int32_t& pb) {
  const int32_t sy = g.nx, sz = g.nx * g.ny;
  pa = x + sy * y + sz * z;
  pb = pa + (axis == 0 ? 1 : (axis == 1 ? sy : sz));
  L.fa = f(x, y, z, pa);
  L.fb = f(x + (axis == 0), y + (axis == 1), z + (axis == 2), pb);
  if (normals) {
    gradient_loads(g, f, x, y, z, L.alo, L.ahi);
    gradient_loads(g, f, x + (axis == 0), y + (axis == 1), z + (axis == 2), L.blo, L.bhi);
  }
}

// Coordinates, unit normal (central differences interpolated along the edge)
// and weight of the point whose field values L holds.
__device__ __forceinline__ void point_finish(const VolGeom& g, int x, int y, int z, int axis,
                                             bool normals, const PointLoads& L, float xyz[3],
                                             float nrm[3], float& w) {
  float ga[3], gb[3];
  if (normals) {
    gradient_finish(g, x, y, z, L.alo, L.ahi, ga);
    gradient_finish(g, x + (axis == 0), y + (axis == 1), z + (axis == 2), L.blo, L.bhi, gb);
  }
  w = (g.iso - L.fa) / (L.fb - L.fa);
  const int ca[3] = {x, y, z};
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const float a = g.origin[d] + g.spacing[d] * (float)ca[d];
    const float b = g.origin[d] + g.spacing[d] * (float)(ca[d] + (d == axis ? 1 : 0));
    xyz[d] = a + w * (b - a);
  }
  if (normals) {
    float m[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) m[d] = ga[d] + w * (gb[d] - ga[d]);
    const float len2 = m[0] * m[0] + m[1] * m[1] + m[2] * m[2];
    if (len2 > 0.0f) {
      const float len = sqrtf(len2);
#pragma unroll
      for (int d = 0; d < 3; ++d) nrm[d] = m[d] / len;
    } else {
      nrm[0] = nrm[1] = nrm[2] = 0.0f;
    }
  }
}

// One interpolated point on the edge with lower endpoint (x,y,z) along axis.
template <class Src>
__device__ __forceinline__ void emit_point(const VolGeom& g, const Src& f, int x, int y, int z,
                                           int axis, bool normals, float xyz[3], float nrm[3],
                                           float& w, int32_t& pa, int32_t& pb) {
  PointLoads L;
  point_loads(g, f, x, y, z, axis, normals, L, pa, pb);
  point_finish(g, x, y, z, axis, normals, L, xyz, nrm, w);
}

// index i with s[i] <= v < s[i+1], s[0..n]
__device__ __forceinline__ int find_word(const uint32_t* s, int n, uint32_t v) {
  int lo = 0, hi = n;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (s[mid] <= v)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

// Edge codes of the 12 cell edges, 5 bits each (edge_code).
__host__ __device__ constexpr uint64_t edge_codes_packed() {
  uint64_t r = 0;
  for (int e = 0; e < 12; ++e) r |= (uint64_t)edge_code(e) << (5 * e);
  return r;
}
constexpr uint64_t kEdgeCodes = edge_codes_packed();

// ---------------------------------------------------------------------------
// Dispatch order of the generate tiles: tiles of class 0 first, then class 1,
// then class 2, each in index order, from a class byte per tile.
constexpr uint32_t kOrderHasOutput = 0x80000000u;  // order entry flag: class 0 or 1

// A thread of the ordering block owns a chunk of K consecutive tiles.  Up to
// kOrderRegTiles of them have their classes loaded before the scan, two bits
// each in a register (the latencies overlap the scan's): byte loads for K
// up to 8, 4-byte loads for K a multiple of 4 up to 32.  Larger chunks (K a
// multiple of 16, volumes of more than 2^28 points) read their class bytes
// in 16-byte vectors while the order is written.  The class arrays end in
// 16 bytes of padding.
constexpr int kOrderRegTiles = 32;
__device__ __forceinline__ uint32_t order_chunk(uint32_t ntl, uint32_t threads) {
  const uint32_t k = (ntl + threads - 1) / threads;
  return k <= 8u ? k : (k <= (uint32_t)kOrderRegTiles ? (k + 3u) / 4u * 4u : (k + 15u) / 16u * 16u);
}
// The loads are unconditional (an address outside the thread's tiles is
// replaced by the first byte, its value dropped), so they issue together
// instead of one conditional load and wait at a time.
__device__ __forceinline__ uint64_t load_classes(const uint8_t* __restrict__ cls, uint32_t t0,
                                                 uint32_t K, uint32_t ntl) {
  uint64_t r = 0ull;
  if (K <= 8u) {
    uint32_t b[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const bool ok = (uint32_t)k < K && t0 + k < ntl;
      b[k] = cls[ok ? t0 + k : 0u];
      b[k] = ok ? b[k] : 0u;
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) r |= (uint64_t)(b[k] & 3u) << (2 * k);
  } else if (K <= (uint32_t)kOrderRegTiles) {
    uint32_t w[kOrderRegTiles / 4];
#pragma unroll
    for (int v = 0; v < kOrderRegTiles / 4; ++v) {
      const uint32_t t = t0 + 4u * v;
      const bool ok = 4u * v < K && t < ntl;  // t0 and K multiples of 4: aligned
      w[v] = *reinterpret_cast<const uint32_t*>(cls + (ok ? t : 0u));
      w[v] = ok ? w[v] : 0u;
    }
#pragma unroll
    for (int v = 0; v < kOrderRegTiles / 4; ++v)
#pragma unroll
      for (int j = 0; j < 4; ++j) r |= (uint64_t)((w[v] >> (8 * j)) & 3u) << (2 * (4 * v + j));
  }
  return r;
}

// Exclusive block scans of two counts per thread (all threads call it; s_a
// and s_b hold a word per wave).
__device__ __forceinline__ void block_scan2(uint32_t a, uint32_t b, uint32_t& ea, uint32_t& eb,
                                            uint32_t& ta, uint32_t& tb, uint32_t* s_a,
                                            uint32_t* s_b) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const uint32_t ia = wave_incl_scan(a), ib = wave_incl_scan(b);
  if (lane == 63) {
    s_a[wv] = ia;
    s_b[wv] = ib;
  }
  __syncthreads();
  uint32_t oa = 0u, ob = 0u;
  ta = tb = 0u;
  const int nwv = (int)(blockDim.x >> 6);
  for (int q = 0; q < nwv; ++q) {
    if (q < wv) {
      oa += s_a[q];
      ob += s_b[q];
    }
    ta += s_a[q];
    tb += s_b[q];
  }
  __syncthreads();  // s_a / s_b reusable
  ea = oa + ia - a;
  eb = ob + ib - b;
}

// Calls fn(k, class) for the thread's tiles k = 0 .. n-1 in order: from reg
// (K <= kOrderRegTiles) or from the class bytes at cls + t0.
template <bool LARGE, class Fn>
__device__ __forceinline__ void for_classes(uint64_t reg, const uint8_t* __restrict__ cls,
                                            uint32_t t0, uint32_t K, uint32_t n, Fn&& fn) {
  if (!LARGE || K <= (uint32_t)kOrderRegTiles) {
    for (uint32_t k = 0; k < n; ++k) fn(k, (uint32_t)(reg >> (2 * k)) & 3u);
    return;
  }
  for (uint32_t v = 0; v < n; v += 16u) {
    const uint4 q = *reinterpret_cast<const uint4*>(cls + t0 + v);
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int j = 0; j < 16; ++j)
      if (v + j < n) fn(v + j, (w[j >> 2] >> (8 * (j & 3))) & 3u);
  }
}

// The next slot of class c's run (cursors s0, s1, s2), in selects and adds:
// a conditional post-increment of one of three cursors is lowered to a
// dynamically indexed private array, one scratch round trip per tile.
__device__ __forceinline__ uint32_t next_slot(uint32_t c, uint32_t& s0, uint32_t& s1,
                                              uint32_t& s2) {
  const uint32_t slot = c == 0u ? s0 : (c == 1u ? s1 : s2);
  s0 += c == 0u ? 1u : 0u;
  s1 += c == 1u ? 1u : 0u;
  s2 += c >= 2u ? 1u : 0u;
  return slot;
}

// Stores order[1 + slot] = v for the (slot, v) pairs that emit_all(put)
// passes to put (every slot in [0, n) once).  Scattered 4-byte stores of
// one block all go through one CU's address unit, a cache line at a time
// (a 16384-entry order took ~10 us); with s_stage (LDS of `stage` entries)
// the pairs are placed in LDS one window of slots at a time, emit_all
// running once per window, and each window leaves in coalesced stores.
// Without s_stage the pairs go straight to global memory.
template <class EmitAll>
__device__ __forceinline__ void store_order(uint32_t* order, uint32_t n, uint32_t* s_stage,
                                            uint32_t stage, EmitAll&& emit_all) {
  if (s_stage == nullptr) {
    emit_all([&](uint32_t slot, uint32_t v) { order[1u + slot] = v; });
    return;
  }
  for (uint32_t lo = 0; lo < n; lo += stage) {
    emit_all([&](uint32_t slot, uint32_t v) {
      if (slot - lo < stage) s_stage[slot - lo] = v;
    });
    __syncthreads();
    const uint32_t m = min(stage, n - lo);
    for (uint32_t i = threadIdx.x; i < m; i += blockDim.x) order[1u + lo + i] = s_stage[i];
    __syncthreads();
  }
}

// order[1 ..] = tiles [0, ntl) of class 0, then 1, then 2, each by index,
// flagged kOrderHasOutput in classes 0 and 1; order[0] = tag.  The thread
// owns tiles [tid * K, tid * K + K).  s_stage may alias s_a and s_b.
template <bool LARGE>
__device__ __forceinline__ void write_order(uint64_t reg, const uint8_t* __restrict__ cls,
                                            uint32_t K, uint32_t ntl, uint32_t* order,
                                            uint32_t tag, uint32_t* s_a, uint32_t* s_b,
                                            uint32_t* s_stage = nullptr, uint32_t stage = 0u) {
  const uint32_t t0 = (uint32_t)threadIdx.x * K;
  const uint32_t n = t0 < ntl ? min(K, ntl - t0) : 0u;
  uint32_t c0 = 0u, c1 = 0u;
  for_classes<LARGE>(reg, cls, t0, K, n, [&](uint32_t, uint32_t c) {
    c0 += c == 0u;
    c1 += c == 1u;
  });
  uint32_t e0, e1, tot0, tot1;
  block_scan2(c0, c1, e0, e1, tot0, tot1, s_a, s_b);
  const uint32_t b0 = e0, b1 = tot0 + e1, b2 = tot0 + tot1 + (t0 - e0 - e1);
  store_order(order, ntl, s_stage, stage, [&](auto&& put) {
    uint32_t s0 = b0, s1 = b1, s2 = b2;
    for_classes<LARGE>(reg, cls, t0, K, n, [&](uint32_t k, uint32_t c) {
      put(next_slot(c, s0, s1, s2), (t0 + k) | (c < 2u ? kOrderHasOutput : 0u));
    });
  });
  if (threadIdx.x == 0) order[0] = tag;
}

// The same order over units of G tiles that lie a plane apart: unit u =
// zg * sp + r (sp tiles per plane) holds tiles (G zg + m) sp + r, m < G,
// and takes the lowest class of its tiles.  The unit of rank R puts its
// tiles at positions 8 G (R / 8) + R % 8 + 8 m: blocks go to the XCDs
// round robin, so a unit's tiles run on one XCD, in consecutive rounds, and
// the field planes they share (three of four for neighbouring planes) are
// fetched into that XCD's L2 once.  Needs every unit whole and nunits a
// multiple of 8; K G <= kOrderRegTiles (the tile classes are loaded before
// the scan, two bits each, by load_unit_classes).
constexpr uint32_t kOrderUnitTiles = 2;  // G
__device__ __forceinline__ uint64_t load_unit_classes(const uint8_t* __restrict__ cls, uint32_t K,
                                                      uint32_t nunits, uint32_t sp) {
  constexpr uint32_t G = kOrderUnitTiles;
  const uint32_t u0 = (uint32_t)threadIdx.x * K;
  const uint32_t n = u0 < nunits ? min(K, nunits - u0) : 0u;
  uint32_t zg = n ? u0 / sp : 0u, r = n ? u0 - zg * sp : 0u;
  uint32_t c[kOrderRegTiles];  // unconditional loads, as in load_classes
#pragma unroll
  for (int k = 0; k < kOrderRegTiles / (int)G; ++k) {
    const bool ok = (uint32_t)k < n;
#pragma unroll
    for (uint32_t m = 0; m < G; ++m) {
      c[k * G + m] = cls[ok ? (G * zg + m) * sp + r : 0u];
      c[k * G + m] = ok ? c[k * G + m] : 0u;
    }
    if (++r == sp) {
      r = 0u;
      ++zg;
    }
  }
  uint64_t reg = 0ull;  // class of tile m of unit k at bits 2 (k G + m)
#pragma unroll
  for (int k = 0; k < kOrderRegTiles; ++k) reg |= (uint64_t)(c[k] & 3u) << (2 * k);
  return reg;
}
__device__ __forceinline__ void write_order_units(uint64_t reg, uint32_t K, uint32_t nunits,
                                                  uint32_t sp, uint32_t* order, uint32_t tag,
                                                  uint32_t* s_a, uint32_t* s_b,
                                                  uint32_t* s_stage = nullptr,
                                                  uint32_t stage = 0u) {
  constexpr uint32_t G = kOrderUnitTiles;
  const uint32_t u0 = (uint32_t)threadIdx.x * K;
  const uint32_t n = u0 < nunits ? min(K, nunits - u0) : 0u;
  auto unit_class = [&](uint32_t k) {
    uint32_t c = 3u;
#pragma unroll
    for (uint32_t m = 0; m < G; ++m) c = min(c, (uint32_t)(reg >> (2u * (k * G + m))) & 3u);
    return c;
  };
  uint32_t c0 = 0u, c1 = 0u;
  for (uint32_t k = 0; k < n; ++k) {
    const uint32_t c = unit_class(k);
    c0 += c == 0u;
    c1 += c == 1u;
  }
  uint32_t e0, e1, tot0, tot1;
  block_scan2(c0, c1, e0, e1, tot0, tot1, s_a, s_b);
  const uint32_t b0 = e0, b1 = tot0 + e1, b2 = tot0 + tot1 + (u0 - e0 - e1);
  store_order(order, nunits * G, s_stage, stage, [&](auto&& put) {
    uint32_t s0 = b0, s1 = b1, s2 = b2;
    uint32_t zg = n ? u0 / sp : 0u, r = n ? u0 - zg * sp : 0u;
    for (uint32_t k = 0; k < n; ++k) {
      const uint32_t R = next_slot(unit_class(k), s0, s1, s2);
      const uint32_t base = 8u * G * (R >> 3) + (R & 7u);
#pragma unroll
      for (uint32_t m = 0; m < G; ++m) {
        const uint32_t tc = (uint32_t)(reg >> (2u * (k * G + m))) & 3u;
        put(base + 8u * m, ((G * zg + m) * sp + r) | (tc < 2u ? kOrderHasOutput : 0u));
      }
      if (++r == sp) {
        r = 0u;
        ++zg;
      }
    }
  });
  if (threadIdx.x == 0) order[0] = tag;
}

// What one wave of a generate tile keeps of a round of up to 64 active cells:
// the cells' table entries, the vertex ids of their 12 edges (the bases of
// the four row words their lower endpoints lie in and each edge's rank there,
// at most 194), their first triangle within the round, and the round's
// triangle -> cell map.
struct GenWave {
  uint64_t table[64];
  uint32_t base[4][64];
  uint8_t rank[12][64];
  uint16_t first[64];
  uint16_t cell[64];           // word << 6 | bit
  uint8_t tri_cell[5 * 64];    // at most 5 triangles per cell
  uint8_t word_mark[64];
};

// LDS layout of a generate tile of TW words and NT threads (wpr known at run
// time): bits (3 planes), active cells, vertex bases (2 planes), triangle
// bases, the waves' rounds.
template <int TW, int NT>
struct GenLayout {
  static constexpr int kWaves = NT / 64;
  int segb, segv;
  __host__ __device__ GenLayout(int wpr) : segb(TW + 2 * wpr + 2), segv(TW + wpr + 2) {}
  __host__ __device__ size_t wave_offset() const {
    return ((size_t)(3 * segb + TW) * 8 + (size_t)(2 * segv + TW + 1) * 4 + 7) / 8 * 8;
  }
  __host__ __device__ size_t bytes() const { return wave_offset() + kWaves * sizeof(GenWave); }
};

// Bits b, b+1, ... of the word A followed by the word A1 (b < 64).
__device__ __forceinline__ uint32_t bit_window(uint64_t A, uint64_t A1, int b) {
  const uint32_t d0 = (uint32_t)A, d1 = (uint32_t)(A >> 32), d2 = (uint32_t)A1;
  const bool up = b >= 32;
  return __builtin_amdgcn_alignbit(up ? d2 : d1, up ? d1 : d0, (uint32_t)b & 31u);
}

// Case and edge ranks of the active cell at bit b of a row word.  Rows of words
// r_yz: r00 the cell's own, r10 / r20 one and two rows up, r01 / r11 / r21
// the same a plane up, r02 / r12 two planes up (each with its next word along
// x, 0 past the row's end).  A row without a neighbour in y (z) is passed as
// its own neighbour, so its edges in that direction vanish.  An edge's id is
// the base of its lower endpoint's word plus its rank among the word's
// active edges; the ranks count bits below b only, which are inside the
// grid, so they need no row-end masks, and the endpoint at b + 1 = 64, bit 0
// of the next word, follows the word's last edge in the numbering.  x2: the
// row has a point b + 2.
struct RowPair {
  uint64_t a, a1;  // a word and the next one along x
};
__device__ __forceinline__ uint32_t rank_below(uint64_t a, uint64_t y, uint64_t z, uint64_t m) {
  return (uint32_t)(popc((a ^ (a >> 1)) & m) + popc((a ^ y) & m) + popc((a ^ z) & m));
}
__device__ __forceinline__ int cell_edges(const RowPair& r00, const RowPair& r10,
                                          const RowPair& r20, const RowPair& r01,
                                          const RowPair& r11, uint64_t r21, uint64_t r02,
                                          uint64_t r12, int b, bool x2, uint32_t* id) {
  const uint64_t m = (1ull << b) - 1ull;
  const uint32_t w00 = bit_window(r00.a, r00.a1, b), w10 = bit_window(r10.a, r10.a1, b);
  const uint32_t w01 = bit_window(r01.a, r01.a1, b), w11 = bit_window(r11.a, r11.a1, b);
  const uint32_t w20 = bit_window(r20.a, r20.a1, b), w02 = bit_window(r02, 0ull, b);
  // flags of the points b (bit 0) and b + 1 (bit 1) of a row
  const uint32_t x00 = w00 ^ (w00 >> 1), y00 = w00 ^ w10, z00 = w00 ^ w01;
  const uint32_t x10 = w10 ^ (w10 >> 1), y10 = w10 ^ w20, z10 = w10 ^ w11;
  const uint32_t x01 = w01 ^ (w01 >> 1), y01 = w01 ^ w11, z01 = w01 ^ w02;
  const uint32_t e00 = rank_below(r00.a, r10.a, r01.a, m);
  const uint32_t e10 = rank_below(r10.a, r20.a, r11.a, m);
  const uint32_t e01 = rank_below(r01.a, r11.a, r02, m);
  const uint32_t e11 = rank_below(r11.a, r21, r12, m);
  const uint32_t n00 = e00 + (x00 & 1u) + (y00 & 1u) + (z00 & 1u);  // first rank at b + 1
  const uint32_t n10 = e10 + (x10 & 1u) + (y10 & 1u) + (z10 & 1u);
  const uint32_t n01 = e01 + (x01 & 1u) + (y01 & 1u) + (z01 & 1u);
  const uint32_t one = x2 ? 1u : 0u;  // x-edges at b + 1 exist
  const uint32_t t00 = (x00 >> 1) & one, t10 = (x10 >> 1) & one, t01 = (x01 >> 1) & one;
  id[0] = e00;
  id[3] = e00 + (x00 & 1u);
  id[8] = e00 + (x00 & 1u) + (y00 & 1u);
  id[1] = n00 + t00;
  id[9] = n00 + t00 + ((y00 >> 1) & 1u);
  id[2] = e10;
  id[11] = e10 + (x10 & 1u) + (y10 & 1u);
  id[10] = n10 + t10 + ((y10 >> 1) & 1u);
  id[4] = e01;
  id[7] = e01 + (x01 & 1u);
  id[5] = n01 + t01;
  id[6] = e11;
  return (int)((w00 & 3u) | ((w10 & 2u) << 1) | ((w10 & 1u) << 3) | ((w01 & 3u) << 4) |
               ((w11 & 2u) << 5) | ((w11 & 1u) << 7));
}

// The row (0: 00, 1: 10, 2: 01, 3: 11) of each edge's lower endpoint, 2 bits
// per edge in the order cell_edges numbers them.
constexpr uint32_t edge_rows_packed() {
  uint32_t r = 0;
  for (int e = 0; e < 12; ++e) {
    const int c = edge_code(e);
    r |= (uint32_t)(((c >> 1) & 1) | (((c >> 2) & 1) << 1)) << (2 * e);
  }
  return r;
}
constexpr uint32_t kEdgeRows = edge_rows_packed();

// 12 contiguous bytes.
template <class T>
__device__ __forceinline__ void store3(T* p, T a, T b, T c) {
  const T v[3] = {a, b, c};
  __builtin_memcpy(p, v, 12);
}

// Edge flags of the word at LDS index lw of plane sA (its +z plane sC) with
// position p; branch-free (the +x word is read and masked).
__device__ __forceinline__ void lds_flags(const VolGeom& g, const uint64_t* sA, const uint64_t* sC,
                                          int lw, const WordPos& p, uint64_t& fx, uint64_t& fy,
                                          uint64_t& fz) {
  const uint64_t A = sA[lw], A1n = sA[lw + 1], B = sA[lw + g.wpr], C = sC[lw];
  edge_flags(p, A, p.q + 1 < g.wpr ? A1n : 0ull, B, C, fx, fy, fz);
}

// Where the generate kernel takes its word bases from: the count kernel's
// per-word prefixes within their count tiles (lpre, v | t << 16), every count
// tile's prefix within its count block (tloc, v | t << 32; the entry after the
// last tile completes the totals) and the count blocks' exclusive prefixes
// (bpre, the totals after the last); the tiles per block are a power of two.
// In a batch the volume's tiles are ct0, ct0 + 1, ..., and the one after its
// last is the next volume's first.  The adjoint and the per-cell outputs take
// the bases from here too.
struct CountSrc {
  const uint32_t* __restrict__ lpre;
  const unsigned long long* __restrict__ tloc;
  const unsigned long long* __restrict__ bpre;
  int64_t n_ctiles, ct0;
  int tpb_shift;  // log2 of the count tiles per count block (from the control block)
};

__device__ __forceinline__ unsigned long long add_vt(unsigned long long a, unsigned long long b) {
  return (unsigned long long)((uint32_t)a + (uint32_t)b) |
         ((unsigned long long)((uint32_t)(a >> 32) + (uint32_t)(b >> 32)) << 32);
}

// Exclusive vertex / triangle prefix (v | t << 32) of count tile c <= n_ctiles
// of the volume.
__device__ __forceinline__ unsigned long long ctile_prefix(const CountSrc& cs, int64_t c) {
  const int64_t g = cs.ct0 + c;
  return add_vt(cs.bpre[g >> cs.tpb_shift], cs.tloc[g]);
}

// Vertex and triangle base of word w (v | t << 32); past the last count tile
// the totals.  Every load is issued (clamped indices, results selected), so
// that the loads of several words can be in flight together.
__device__ __forceinline__ unsigned long long word_bases(const CountSrc& cs, int64_t w) {
  const int64_t ct = w / kCountTile;
  const bool past = ct >= cs.n_ctiles;
  const unsigned long long p = ctile_prefix(cs, past ? cs.n_ctiles : ct);
  const uint32_t lw = cs.lpre[past ? 0 : w], l = past ? 0u : lw;
  return add_vt(p, (unsigned long long)(l & 0xffffu) | ((unsigned long long)(l >> 16) << 32));
}

// Exclusive scan of the n count-block sums (v | t << 32, each half below
// 2^32) by one block of kTsumThreads threads into bpre, the totals after the
// last: four consecutive sums per thread and round, wave scans of the thread
// totals' halves, the block's wave sums in 64 bits, 64-bit carries between
// rounds.  s_v and s_t hold a word per wave.  Returns the totals in cv, ct.
constexpr int kTsumThreads = 1024;
constexpr int kTsumPerThread = 4;  // block sums per thread and round
__device__ __forceinline__ void scan_block_sums(const unsigned long long* __restrict__ bsum,
                                                unsigned long long* __restrict__ bpre, int64_t n,
                                                uint32_t* s_v, uint32_t* s_t,
                                                unsigned long long& cv, unsigned long long& ct) {
  constexpr int kWaves = kTsumThreads / 64, kPer = kTsumPerThread;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  cv = ct = 0ull;
  for (int64_t e0 = 0; e0 < n; e0 += kPer * kTsumThreads) {
    const int64_t e = e0 + (int64_t)kPer * tid;  // the thread's kPer consecutive sums
    uint32_t v[kPer], t[kPer], sv = 0u, st = 0u;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const unsigned long long x = e + i < n ? bsum[e + i] : 0ull;
      v[i] = (uint32_t)x;
      t[i] = (uint32_t)(x >> 32);
      sv += v[i];
      st += t[i];
    }
    // a round's sums stay below 2^32 only for the wave partials (a count
    // block holds at most 3 * 2^18 vertices); the cross-wave totals are
    // formed in 64 bits
    const uint32_t iv = wave_incl_scan(sv), it = wave_incl_scan(st);
    if (lane == 63) {
      s_v[wv] = iv;
      s_t[wv] = it;
    }
    __syncthreads();
    unsigned long long ov = 0, ot = 0, rv = 0, rt = 0;
#pragma unroll
    for (int q = 0; q < kWaves; ++q) {
      if (q < wv) {
        ov += s_v[q];
        ot += s_t[q];
      }
      rv += s_v[q];
      rt += s_t[q];
    }
    __syncthreads();
    unsigned long long pv = cv + ov + iv - sv, pt = ct + ot + it - st;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      if (e + i < n) bpre[e + i] = (pv & 0xffffffffull) | (pt << 32);
      pv += v[i];
      pt += t[i];
    }
    cv += rv;
    ct += rt;
  }
  if (tid == 0) bpre[n] = (cv & 0xffffffffull) | (ct << 32);
}

// One generate tile: words [w_begin, w_begin + TW) of a volume, a block of NT
// threads.
//   1. stage bits (planes k, k+1, k+2), vertex bases (k, k+1), triangle bases
//   2. a thread per word: active-cell mask.  The last barrier: from here each
//      wave works alone
//   3. a thread per output vertex: word by binary search over the vertex
//      bases, edge by popcount select; coordinates, normal, records
//   4. each wave takes a run of words with its share of the tile's triangles,
//      in rounds of 64 active cells: words mark their first cell's lane, a
//      prefix maximum gives every lane its word and a popcount select its
//      cell; the lane forms the cell's case and the ids of all 12 edges at
//      once (cell_edges: a third of the operations of ranking each triangle
//      corner by itself), then a lane per triangle picks three of them
//
// What bounds it: VALU issue and the chain of loads (staging, then the field
// values of a vertex).  The waves share the staged words but no barriers, so
// the chains of different waves overlap.  A block of 256 threads with rounds
// between barriers took, with 512-word tiles, 63 us at 37 x 29 x 33 points, 86
// at 256^3 (475 K vertices) and 88 at 512^3 (957 K); this one, with the tiles
// gen_shape picks, 13, 36 and 62.
//
// The bases come from the count kernel's prefixes (cs).  has_output skips the
// check for a tile without output (one round trip).
template <int TW, int NT, class Src, bool dedup>
__device__ __forceinline__ void generate_tile(const VolGeom& g, const Src& f,
                                              const uint64_t* __restrict__ b, int64_t w_begin,
                                              const OutPtrs& out, bool normals,
                                              int64_t vol_base_v, int64_t vol_base_t,
                                              uint64_t* s_dyn, const CountSrc& cs,
                                              bool has_output) {
  const int tid = threadIdx.x, lane = tid & 63;
  static_assert(NT >= TW, "a thread per word");
  constexpr int nt = NT, nwaves = NT / 64;
  const int nw = (int)min((int64_t)TW, g.nwords - w_begin);
  if (!has_output) {  // count tiles without output
    const int64_t c0 = w_begin / kCountTile;
    const int64_t c1 = min((w_begin + nw + kCountTile - 1) / kCountTile, cs.n_ctiles);
    if (ctile_prefix(cs, c0) == ctile_prefix(cs, c1)) return;
  }

  const GenLayout<TW, NT> L(g.wpr);
  uint64_t* s_b0 = s_dyn;
  uint64_t* s_b1 = s_b0 + L.segb;
  uint64_t* s_b2 = s_b1 + L.segb;
  uint64_t* s_act = s_b2 + L.segb;
  uint32_t* s_v0 = reinterpret_cast<uint32_t*>(s_act + TW);
  uint32_t* s_v1 = s_v0 + L.segv;
  uint32_t* s_t = s_v1 + L.segv;
  GenWave& W = reinterpret_cast<GenWave*>(reinterpret_cast<char*>(s_dyn) + L.wave_offset())[tid >> 6];

  // staging: each thread issues the loads of up to kStageU of its words
  // (clamped indices, every load unconditional) before storing any of them,
  // so they are in flight together rather than one conditional load and
  // wait at a time
  constexpr int kStageU = 4;
  const int64_t plane = (int64_t)g.wpr * g.ny;
  for (int i0 = tid; i0 < L.segb; i0 += kStageU * nt) {
    uint64_t v[kStageU][3];
#pragma unroll
    for (int u = 0; u < kStageU; ++u) {
      const int64_t w = w_begin + i0 + u * nt;
#pragma unroll
      for (int z = 0; z < 3; ++z) v[u][z] = b[w + z * plane < g.nwords ? w + z * plane : 0];
    }
#pragma unroll
    for (int u = 0; u < kStageU; ++u) {
      const int i = i0 + u * nt;
      if (i < L.segb) {
        const int64_t w = w_begin + i;
        s_b0[i] = (w < g.nwords) ? v[u][0] : 0ull;
        s_b1[i] = (w + plane < g.nwords) ? v[u][1] : 0ull;
        s_b2[i] = (w + 2 * plane < g.nwords) ? v[u][2] : 0ull;
      }
    }
  }
  for (int i0 = tid; i0 < L.segv; i0 += kStageU * nt) {
    unsigned long long p0[kStageU], p1[kStageU];
#pragma unroll
    for (int u = 0; u < kStageU; ++u) {
      const int i = i0 + u * nt;
      p0[u] = word_bases(cs, w_begin + i);
      p1[u] = word_bases(cs, w_begin + plane + i);
    }
#pragma unroll
    for (int u = 0; u < kStageU; ++u) {
      const int i = i0 + u * nt;
      if (i < L.segv) {
        s_v0[i] = (uint32_t)p0[u];
        s_v1[i] = (uint32_t)p1[u];
        if (i <= nw) s_t[i] = (uint32_t)(p0[u] >> 32);
      }
    }
  }
  __syncthreads();
  const uint32_t tv0 = s_v0[0], tv1 = s_v0[nw];
  const uint32_t tt0 = s_t[0], tt1 = s_t[nw];
  if (tv0 == tv1 && tt0 == tt1) return;  // no output here

  // 2. active cells of the thread's word
  if (tid < nw) {
    const WordPos p = word_pos(g, w_begin + tid);
    const bool nx1 = p.q + 1 < g.wpr;
    CellPlanes cp;
    cell_planes(p, s_b0[tid], nx1 ? s_b0[tid + 1] : 0ull, s_b0[tid + g.wpr],
                nx1 ? s_b0[tid + g.wpr + 1] : 0ull, s_b1[tid], nx1 ? s_b1[tid + 1] : 0ull,
                s_b1[tid + g.wpr], nx1 ? s_b1[tid + g.wpr + 1] : 0ull, cp);
    s_act[tid] = cp.active;
  }
  __syncthreads();

  // 3. vertices (dedup: one per active edge, in id order).  A thread's
  //    first vertex is located and its field values loaded here, and
  //    finished after the triangle rounds: the loads' latency overlaps the
  //    rounds' LDS work.
  const int nV = (int)(tv1 - tv0);
  auto locate = [&](int vl, int& x, int& y, int& z, int& axis) {
    const int li = find_word(s_v0, nw, tv0 + (uint32_t)vl);
    const WordPos p = word_pos(g, w_begin + li);
    uint64_t fx, fy, fz;
    lds_flags(g, s_b0, s_b1, li, p, fx, fy, fz);
    int bit;
    edge_select(fx, fy, fz, (int)(tv0 + (uint32_t)vl - s_v0[li]), bit, axis);
    x = p.q * 64 + bit;
    y = p.j;
    z = p.k;
  };
  auto store_vertex = [&](int vl, int axis, const float xyz[3], const float nrm[3], float w,
                          int32_t pa, int32_t pb) {
    const int64_t gv = (int64_t)tv0 + vl;
    store3(out.vertices + 3 * gv, xyz[0], xyz[1], xyz[2]);
    if (normals) store3(out.normals + 3 * gv, nrm[0], nrm[1], nrm[2]);
    if (out.edges) out.edges[gv] = ((uint32_t)axis << 30) | (uint32_t)pa;
    if (out.interp_first) out.interp_first[gv] = (int32_t)pa;
    if (out.interp_second) out.interp_second[gv] = (int32_t)pb;
    if (out.interp_weight) out.interp_weight[gv] = w;
  };
  const bool first = dedup && tid < nV;
  int fx0 = 0, fy0 = 0, fz0 = 0, fax = 0;
  int32_t fpa = 0, fpb = 0;
  PointLoads fl;
  if (first) {
    locate(tid, fx0, fy0, fz0, fax);
    point_loads(g, f, fx0, fy0, fz0, fax, normals, fl, fpa, fpb);
  }

  // 4. triangles: the wave's words are those whose first triangle lies in its
  //    share of the tile's (lanes 0 and 1 search its ends)
  const int n_tri = (int)(tt1 - tt0);
  int wa = 0, wb = nw;
  if constexpr (nwaves > 1) {
    const uint32_t part = (uint32_t)(tid >> 6) + (lane == 1 ? 1u : 0u);
    const uint32_t want = tt0 + part * (uint32_t)n_tri / (uint32_t)nwaves;
    int lo = 0, hi = nw;  // first word whose base is at least `want`
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      const bool below = s_t[mid] < want;
      lo = below ? mid + 1 : lo;
      hi = below ? hi : mid;
    }
    wa = __builtin_amdgcn_readlane(lo, 0);
    wb = part == (uint32_t)nwaves ? nw : lo;
    wb = __builtin_amdgcn_readlane(wb, 1);
  }
  int64_t tri = n_tri > 0 && wa < wb ? (int64_t)s_t[wa] : 0;
  for (int c = wa; c < wb && n_tri > 0; c += 64) {  // wave-uniform
    const uint64_t act_l = c + lane < wb ? s_act[c + lane] : 0ull;
    const uint32_t nc = (uint32_t)popc(act_l);
    const uint32_t inc = wave_incl_scan(nc), n_cells = wave_last(inc), start = inc - nc;
    for (uint32_t c0 = 0; c0 < n_cells; c0 += 64u) {
      W.word_mark[lane] = 0;
      wave_lds_sync();
      if (nc != 0u && start < c0 + 64u && inc > c0)
        W.word_mark[max(start, c0) - c0] = (uint8_t)(lane + 1);
      wave_lds_sync();
      const int wl = (int)wave_incl_max((uint32_t)W.word_mark[lane]) - 1;
      const uint32_t slot = c0 + (uint32_t)lane;
      const bool valid = slot < n_cells;
      const uint32_t wstart = (uint32_t)__shfl((int)start, wl, 64);
      const int li = c + wl;
      const int bit = select_bit(s_act[li], valid ? (int)(slot - wstart) : 0);
      const WordPos p = word_pos(g, w_begin + li);
      const bool nx1 = p.q + 1 < g.wpr, hy2 = p.j + 2 < g.ny, hz2 = p.k + 2 < g.nz;
      const int l1 = li + g.wpr, l2 = hy2 ? l1 + g.wpr : l1;
      const uint64_t* s_z2 = hz2 ? s_b2 : s_b1;
      auto pair = [&](const uint64_t* row, int i) {
        const uint64_t n = row[i + 1];
        return RowPair{row[i], nx1 ? n : 0ull};
      };
      uint32_t id[12];
      const int cs = cell_edges(pair(s_b0, li), pair(s_b0, l1), pair(s_b0, l2), pair(s_b1, li),
                                pair(s_b1, l1), s_b1[l2], s_z2[li], s_z2[l1], bit,
                                p.q * 64 + bit + 2 < g.nx, id);
      const uint64_t table = c_case_table[cs];
      const uint32_t nf = valid ? (uint32_t)(table >> 60) : 0u;
      const uint32_t finc = wave_incl_scan(nf), round_tris = wave_last(finc), ffirst = finc - nf;
      W.table[lane] = table;
      W.first[lane] = (uint16_t)ffirst;
      if (dedup) {
        W.base[0][lane] = s_v0[li];
        W.base[1][lane] = s_v0[l1];
        W.base[2][lane] = s_v1[li];
        W.base[3][lane] = s_v1[l1];
#pragma unroll
        for (int e = 0; e < 12; ++e) W.rank[e][lane] = (uint8_t)id[e];
      } else {
        W.cell[lane] = (uint16_t)((li << 6) | bit);
      }
#pragma unroll
      for (uint32_t t = 0; t < 5u; ++t)
        if (t < nf) W.tri_cell[ffirst + t] = (uint8_t)lane;
      wave_lds_sync();
      for (uint32_t tl = (uint32_t)lane; tl < round_tris; tl += 64u) {
        const int cl = (int)W.tri_cell[tl];
        const uint32_t visit = tl - W.first[cl];
        const uint32_t es = (uint32_t)(W.table[cl] >> (12u * visit));
        const int64_t t = tri + tl;
        int32_t ids[3];
        if (dedup) {
#pragma unroll
          for (int v = 0; v < 3; ++v) {
            const uint32_t e = (es >> (4 * v)) & 15u;
            ids[v] = (int32_t)((int64_t)W.base[(kEdgeRows >> (2u * e)) & 3u][cl] + W.rank[e][cl] -
                               vol_base_v);
          }
        } else {
          const int cw = (int)W.cell[cl] >> 6, cb = (int)W.cell[cl] & 63;
          const WordPos pc = word_pos(g, w_begin + cw);
#pragma unroll
          for (int v = 0; v < 3; ++v) {
            const int code = (int)((kEdgeCodes >> (5 * ((es >> (4 * v)) & 15u))) & 31u);
            const int64_t corner = 3 * t + v;
            float xyz[3], nrm[3], w;
            int32_t pa, pb;
            emit_point(g, f, pc.q * 64 + cb + (code & 1), pc.j + ((code >> 1) & 1),
                       pc.k + ((code >> 2) & 1), code >> 3, normals, xyz, nrm, w, pa, pb);
            store3(out.vertices + 3 * corner, xyz[0], xyz[1], xyz[2]);
            if (normals) store3(out.normals + 3 * corner, nrm[0], nrm[1], nrm[2]);
            if (out.interp_first) out.interp_first[corner] = (int32_t)pa;
            if (out.interp_second) out.interp_second[corner] = (int32_t)pb;
            if (out.interp_weight) out.interp_weight[corner] = w;
            ids[v] = (int32_t)(corner - 3 * vol_base_t);
          }
        }
        store3(out.conn + 3 * t, ids[0], ids[1], ids[2]);
      }
      tri += round_tris;
      wave_lds_sync();  // the round's LDS is reused
    }
  }

  if (first) {
    float xyz[3], nrm[3], w;
    point_finish(g, fx0, fy0, fz0, fax, normals, fl, xyz, nrm, w);
    store_vertex(tid, fax, xyz, nrm, w, fpa, fpb);
  }
  if (dedup) {
    for (int vl = tid + nt; vl < nV; vl += nt) {
      int x, y, z, axis;
      locate(vl, x, y, z, axis);
      float xyz[3], nrm[3], w;
      int32_t pa, pb;
      emit_point(g, f, x, y, z, axis, normals, xyz, nrm, w, pa, pb);
      store_vertex(vl, axis, xyz, nrm, w, pa, pb);
    }
  }
}

}  // namespace mc
}  // namespace daxhip
