// Device code of the marching-cubes adjoint, shared by the single-volume
// and the batched backward.
//
// Forward, per output vertex u on the active edge (A, B = A + e_axis):
//   t   = (iso - fA) / (fB - fA)
//   x_u = cA + t (cB - cA)                       (Lerp of the corner coordinates)
//   m   = gA + t (gB - gA),  n_u = m / |m|       (g: central-difference gradient)
// Topology (which edges are active) is held piecewise constant.  Given
// dL/dx_u and dL/dn_u the adjoint is
//   dL/dm = (dL/dn - n (n . dL/dn)) / |m|
//   dL/dt = dL/dx . (cB - cA) + dL/dm . (gB - gA)
//   dL/dfA += dL/dt * (-(1-t)/(fB-fA)),   dL/dfB += dL/dt * (-t/(fB-fA))
//   dL/dgA  = (1-t) dL/dm,                dL/dgB  = t dL/dm
// and each dL/dg_p[d] flows to the stencil points of g_p[d].
//
// Deterministic (no atomics; every sum has a fixed order), in four launches
// (three where the endpoints add up the few tiles' counts themselves):
//   records    one thread per vertex, recomputes t, gA, gB from the field and
//              the compact edge list (the interpolants are not stored by the
//              forward), writes 8 floats per vertex (sA, GA[3], sB, GB[3]);
//              beside it the row words' endpoints are written
//              (the points of active edges) and their counts, a wave per tile
//   scan       the tiles' endpoint counts, so that every endpoint has a slot
//   endpoints  each endpoint's sums (S, G) over its at most 6 edges, once
//   gather     every point: 0, or within L1 distance 1 of an endpoint (the
//              only points with a non-zero dL/df) the sum of its own S and the
//              stencil terms of the G of its neighbours
#pragma once

#include <algorithm>

#include "mc_kernels.h"

namespace daxhip {
namespace mc {

// Per-vertex adjoint record: the lower endpoint's half and the upper
// endpoint's half, 16 bytes each.
struct alignas(16) VertexAdj {
  float sA, gA[3], sB, gB[3];
};
static_assert(sizeof(VertexAdj) == 32, "32-byte vertex records");

__device__ __forceinline__ void grad_at(const VolGeom& g, const float* f, int x, int y, int z,
                                        float out[3]) {
  // branch-free loads (point_gradient): the six values of a gradient, and
  // both gradients of a vertex, are in flight together
  point_gradient(g, FieldArray{f}, x, y, z, out);
}

// Adjoint record of vertex u (global index into edges/dldx/dldn/out) of the
// volume g; the edge code is local to the volume.
__device__ __forceinline__ void vertex_adjoint(const VolGeom& g, const float* __restrict__ field,
                                               const uint32_t* __restrict__ edges,
                                               const float* __restrict__ dldx,
                                               const float* __restrict__ dldn, int64_t u,
                                               VertexAdj* __restrict__ out) {
  const float* f = field + g.field_off;
  const uint32_t e = edges[u];
  const int axis = (int)(e >> 30);
  const int64_t A = (int64_t)(e & 0x3fffffffu);
  const int64_t sy = g.nx, sz = (int64_t)g.nx * g.ny;
  const uint32_t A32 = (uint32_t)A, row = fast_div(A32, g.div_nx);  // A < 2^30
  const uint32_t zz = fast_div(row, g.div_ny);
  const int x = (int)(A32 - row * (uint32_t)g.nx), y = (int)(row - zz * (uint32_t)g.ny),
            z = (int)zz;
  // an edge code outside the grid (edge list not written by a forward that
  // fit its outputs) contributes nothing and is never dereferenced
  if (axis > 2 || A >= sz * g.nz || x + (axis == 0) >= g.nx || y + (axis == 1) >= g.ny ||
      z + (axis == 2) >= g.nz) {
    out[u] = VertexAdj{0.0f, {0.0f, 0.0f, 0.0f}, 0.0f, {0.0f, 0.0f, 0.0f}};
    return;
  }
  const int64_t B = A + (axis == 0 ? 1 : (axis == 1 ? sy : sz));
  // the upstream gradients do not depend on the field: load them first
  const float dn[3] = {dldn[3 * u + 0], dldn[3 * u + 1], dldn[3 * u + 2]};
  const float dx[3] = {dldx[3 * u + 0], dldx[3 * u + 1], dldx[3 * u + 2]};
  const float fA = f[A], fB = f[B];
  const float den = fB - fA;
  const float t = (g.iso - fA) / den;
  float gA[3], gB[3];
  grad_at(g, f, x, y, z, gA);
  grad_at(g, f, x + (axis == 0), y + (axis == 1), z + (axis == 2), gB);
  float m[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) m[d] = gA[d] + t * (gB[d] - gA[d]);
  const float len2 = m[0] * m[0] + m[1] * m[1] + m[2] * m[2];
  float dm[3] = {0.0f, 0.0f, 0.0f};
  if (len2 > 0.0f) {
    const float len = sqrtf(len2);
    float nv[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) nv[d] = m[d] / len;
    const float dot = nv[0] * dn[0] + nv[1] * dn[1] + nv[2] * dn[2];
#pragma unroll
    for (int d = 0; d < 3; ++d) dm[d] = (dn[d] - nv[d] * dot) / len;
  }
  const int ca[3] = {x, y, z};
  float dldt = 0.0f;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const float a = g.origin[d] + g.spacing[d] * (float)ca[d];
    const float b = g.origin[d] + g.spacing[d] * (float)(ca[d] + (d == axis ? 1 : 0));
    dldt += dx[d] * (b - a);
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) dldt += dm[d] * (gB[d] - gA[d]);
  VertexAdj r;
  r.sA = dldt * (-(1.0f - t) / den);
  r.sB = dldt * (-t / den);
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    r.gA[d] = (1.0f - t) * dm[d];
    r.gB[d] = t * dm[d];
  }
  out[u] = r;
}

// ---- endpoints and gather ---------------------------------------------------
// Endpoint words and prefixes a wave per tile of 256 row words, sums and gather
// a wave per WW words; nothing is shared between the waves of a block.  What the
// steps hand on goes through global memory (the caches), so a wave needs
// little LDS and no barrier, and no work is repeated at tile borders.  A block
// per tile that staged edge flags with a halo, formed the sums of the tile's
// and the halo's endpoints in LDS between six barriers and listed tiles too
// dense for it for another pass took 56 + 28 us at 256^3 (447 K endpoints),
// 490 + 14 on a noisy 640^3 surface (3.6 M), 375 + 60 for 256 volumes of
// 32..160 points an axis (1.4 M) and 1674 + 4 on the 1024^3 Mandelbulb.  Sums and
// gather take 20 + 24, 100 + 311, 57 + 264 and 252 + 1216; the words, beside the
// records, and their scan 4, 30, 28 and 105 more.
constexpr int kAdjTile = kGatherTileWords;  // row words per tile
constexpr int kAdjThreads = kAdjTile;
// Words per wave of the sums and the gather (adjoint_wave_words).
template <int WW>
constexpr int kAdjBlockWords = kAdjThreads / 64 * WW;
template <int WW>
constexpr int kAdjTileBlocks = kAdjTile / kAdjBlockWords<WW>;
// Waves per SIMD the gather is compiled for: as many as there are, except on
// large volumes, where fewer waves keep what they share in the caches (1024^3
// 1258 us with 8, 1216 with the 6 it takes by itself; 256 volumes 279, 264).
template <int WW>
constexpr int kGatherWaves = WW == 64 ? 1 : 8;

// How many edges of the list a call takes: n_points, and not more than counts[1]
// where the forward's counts are given.
struct EdgeList {
  const int64_t* counts;
  int64_t n_points;
};
__device__ __forceinline__ int64_t edge_count(const EdgeList& l) {
  return l.counts ? min(l.counts[1], l.n_points) : l.n_points;
}

// Endpoint words of a volume (or batch) and their prefixes: the endpoints of
// word w before it are tile[w's tile] + pre[w].
struct Endpoints {
  uint64_t* words;
  uint16_t* pre;
  uint32_t* sums;  // per tile
  uint32_t* tile;  // their exclusive prefixes
  uint32_t* base;  // per count tile: vertex base
};
static_assert(kAdjTile * 64 < 65536, "prefixes within a tile fit 16 bits");
static_assert(kAdjTile == 2 * kCountTile, "two count tiles per tile");

// Vertex base of row word w of a volume (lpre: its count prefixes).
__device__ __forceinline__ uint32_t vertex_base(const VolGeom& g, const Endpoints& ep,
                                                const uint32_t* __restrict__ lpre, int64_t w) {
  return ep.base[2 * g.tile_off + w / kCountTile] + (lpre[w] & 0xffffu);
}

// Endpoint words, counts and prefixes of a tile by one wave, four consecutive
// words a lane.  Endpoints of a word: the points whose bit differs from one of
// their neighbours' (grids without cells have none).  They depend on the bits
// alone, not on how many of the edges a call takes, so that calls that share a
// workspace write the same values there.
__device__ __forceinline__ void endpoint_words_tile(const VolGeom& g,
                                                    const uint64_t* __restrict__ b,
                                                    const CountSrc& cs, const Endpoints& ep,
                                                    int64_t w0) {
  const int lane = threadIdx.x & 63;
  const int64_t w = w0 + 4 * lane, plane = (int64_t)g.wpr * g.ny;
  const int64_t tile = g.tile_off + w0 / kAdjTile;
  uint64_t e[4] = {0ull, 0ull, 0ull, 0ull};
  uint32_t n = 0u;
  if (w < g.nwords) {
    auto load4 = [&](int64_t at, uint64_t (&v)[4]) {
      if (at >= 0 && at + 4 <= g.nwords) {
        __builtin_memcpy(v, b + at, 32);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = at + i >= 0 && at + i < g.nwords ? b[at + i] : 0ull;
      }
    };
    uint64_t A[4], yp[4], ym[4], zp[4], zm[4];
    load4(w, A);
    load4(w + g.wpr, yp);
    load4(w - g.wpr, ym);
    load4(w + plane, zp);
    load4(w - plane, zm);
    uint64_t prev = w > 0 ? b[w - 1] : 0ull;
    const uint64_t last = w + 4 < g.nwords ? b[w + 4] : 0ull;
    WordIter wi;
    wi.init(g, (int)w);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const WordPos p = wi.pos(g);
      const uint64_t a = A[i], next = p.q + 1 < g.wpr ? (i < 3 ? A[(i + 1) % 4] : last) : 0ull;
      const uint64_t fx = (a ^ shr1(a, next)) & p.xmask;
      uint64_t m = fx | (fx << 1);
      if (p.q > 0) m |= ((prev >> 63) ^ a) & 1ull;
      if (p.has_y) m |= a ^ yp[i];
      if (p.j > 0) m |= a ^ ym[i];
      if (p.has_z) m |= a ^ zp[i];
      if (p.k > 0) m |= a ^ zm[i];
      e[i] = w + i < g.nwords ? m & p.pmask : 0ull;
      n += (uint32_t)popc(e[i]);
      prev = a;
      wi.next(g);
    }
  }
  const uint32_t inc = wave_incl_scan(n);
  uint32_t run = inc - n;
  uint16_t pre[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    pre[i] = (uint16_t)run;
    run += (uint32_t)popc(e[i]);
  }
  if (w + 4 <= g.nwords) {
    __builtin_memcpy(ep.words + g.word_off + w, e, 32);
    __builtin_memcpy(ep.pre + g.word_off + w, pre, 8);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (w + i < g.nwords) {
        ep.words[g.word_off + w + i] = e[i];
        ep.pre[g.word_off + w + i] = pre[i];
      }
  }
  if (lane == 63) ep.sums[tile] = inc;
  if (lane < 2) {
    const int64_t c = w0 / kCountTile + lane;
    if (c < cs.n_ctiles) ep.base[2 * g.tile_off + c] = (uint32_t)ctile_prefix(cs, c);
  }
}

// Exclusive scan of the tiles' counts, a block per kScanTiles of them (at most
// kScanBlocks blocks, so more each for more tiles): a block sums up what lies
// before its part by itself.  It also clears slot 0 of the endpoints' sums,
// which stands for the points that are no endpoints.
constexpr int kAdjScanThreads = 1024;
constexpr int64_t kScanTiles = (int64_t)kAdjScanThreads * kScanChunk;
constexpr int kScanBlocks = 16;
static __global__ __launch_bounds__(kAdjScanThreads) void k_scan_endpoints(
    const uint32_t* __restrict__ sums, uint32_t* __restrict__ pre, int64_t n, int64_t part,
    EdgeList list, f32x4* __restrict__ endpoint_sums) {
  __shared__ uint32_t s_scan[kAdjScanThreads / 64];
  if (blockIdx.x == 0 && threadIdx.x == 0) endpoint_sums[0] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  if (edge_count(list) == 0) return;
  const int64_t first = (int64_t)blockIdx.x * part, end = min(first + part, n);
  uint32_t before = 0u, carry;
  for (int64_t i = 4 * (int64_t)threadIdx.x; i < first; i += 4 * kAdjScanThreads) {
    uint32_t v[4];  // first is a multiple of 4
    __builtin_memcpy(v, sums + i, 16);
    before += v[0] + v[1] + v[2] + v[3];
  }
  (void)block_excl_scan(before, carry, s_scan);
  for (int64_t c0 = first; c0 < end; c0 += kScanTiles) {
    const int64_t i0 = c0 + (int64_t)threadIdx.x * kScanChunk;
    u32x4 x[kScanChunk / 4];
    load_chunk(sums, i0, n, x);
    uint32_t sum = 0u, total;
#pragma unroll
    for (int q = 0; q < kScanChunk; ++q) sum += x[q / 4][q % 4];
    const uint32_t run = carry + block_excl_scan(sum, total, s_scan);
    carry += total;
    store_prefixes(pre, i0, n, x, run);
  }
}
inline int launch_scan_endpoints(const Endpoints& ep, int64_t tiles, const EdgeList& list,
                                 f32x4* sums, hipStream_t s) {
  const int64_t part = align_up(
      (size_t)std::max(kScanTiles, ceil_div(tiles, (int64_t)kScanBlocks)), (size_t)kScanTiles);
  k_scan_endpoints<<<dim3((unsigned)ceil_div(tiles, part)), kAdjScanThreads, 0, s>>>(
      ep.sums, ep.tile, tiles, part, list, sums);
  DAXHIP_LAUNCH_CHECK("k_scan_endpoints");
  return DAX_HIP_OK;
}

// Up to this many tiles the sums' blocks add up the counts before their tile
// themselves and leave them for the gather, which saves the scan's launch.
constexpr int64_t kFoldTiles = 1024;

// Endpoints before `tile`: from the scan, or (fold) the counts' sum (all threads
// of the block, whose first one notes it for the gather).
template <bool FOLD>
__device__ __forceinline__ uint32_t endpoints_before(const Endpoints& ep, int64_t tile, bool note,
                                                     const EdgeList& list) {
  if constexpr (!FOLD) return ep.tile[tile];
  __shared__ uint32_t s_sum[kAdjThreads / 64];
  uint32_t v = 0u;
#pragma unroll
  for (int u = 0; u < (int)(kFoldTiles / kAdjThreads); ++u) {
    const int i = u * kAdjThreads + (int)threadIdx.x;
    v += i < tile ? ep.sums[i] : 0u;
  }
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) s_sum[threadIdx.x >> 6] = v;
  __syncthreads();
  v = 0u;
#pragma unroll
  for (int q = 0; q < kAdjThreads / 64; ++q) v += s_sum[q];
  if (note && threadIdx.x == 0 && edge_count(list) != 0) ep.tile[tile] = v;
  return v;
}

__device__ __forceinline__ uint64_t shfl64(uint64_t v, int l) {
  return ((uint64_t)(uint32_t)__shfl((int)(uint32_t)(v >> 32), l, 64) << 32) |
         (uint32_t)__shfl((int)(uint32_t)v, l, 64);
}

// The lane's word among lanes holding n items each (inclusive scan inc), for
// the 64 items from e0 on: words mark their first item's lane, a prefix
// maximum gives every lane its word.  Lanes past the last item get the last
// word.
__device__ __forceinline__ int item_word(uint32_t n, uint32_t inc, uint32_t e0, uint8_t* mark) {
  const int lane = threadIdx.x & 63;
  const uint32_t start = inc - n;
  mark[lane] = 0;
  wave_lds_sync();
  if (n != 0u && start < e0 + 64u && inc > e0) mark[max(start, e0) - e0] = (uint8_t)(lane + 1);
  wave_lds_sync();
  const int wl = (int)wave_incl_max((uint32_t)mark[lane]) - 1;
  wave_lds_sync();  // the marks are reused
  return wl;
}

// (S_p, dL/dg_p) of the endpoint p at `bit` of row word w: over the 3 edges
// leaving p (lower halves of their records), then the 3 edges entering p
// (upper halves), in axis order.  The edges leaving p follow each other in
// the numbering, the x-edge entering it is counted back from them; the y- and
// z-edges entering it are ranked in their own words.  Words are shifted up so
// that p's bit is their sign and the bits above it are gone: a flag is then a
// comparison, and the edges of the points up to p are popcounts.
__device__ __forceinline__ f32x4 endpoint_sums(const VolGeom& g, const uint64_t* __restrict__ b,
                                               const uint32_t* __restrict__ lpre,
                                               const Endpoints& ep,
                                               const VertexAdj* __restrict__ adj, int64_t n_adj,
                                               int64_t w, int bit) {
  const int64_t plane = (int64_t)g.wpr * g.ny;
  const WordPos p = word_pos(g, w);
  const bool hn = p.q + 1 < g.wpr;
  const int up = 63 - bit;
  // rows: own, +y, +z; the row before with +z; the plane before with +y (a row
  // that is not there: one without edges to it)
  const int64_t wy = p.j > 0 ? w - g.wpr : w, wz = p.k > 0 ? w - plane : w;
  const int64_t sy = p.has_y ? g.wpr : 0, sz = p.has_z ? plane : 0;
  const uint64_t A0 = b[w], Y0 = b[wy], Z0 = b[wz];
  const uint64_t An = hn ? b[w + 1] : 0ull, Yn = hn ? b[wy + 1] : 0ull, Zn = hn ? b[wz + 1] : 0ull;
  const uint64_t B = b[w + sy] << up, C = b[w + sz] << up;
  const uint64_t YC = b[wy + sz] << up, ZB = b[wz + sy] << up;
  const uint32_t ba = vertex_base(g, ep, lpre, w), by = vertex_base(g, ep, lpre, wy),
                 bz = vertex_base(g, ep, lpre, wz);
  const uint64_t A = A0 << up, Y = Y0 << up, Z = Z0 << up;
  auto sign = [](uint64_t v) -> uint32_t { return (uint32_t)(v >> 32) >> 31; };
  const uint32_t xin = p.q * 64 + bit + 1 < g.nx ? 1u : 0u;  // an x-edge leaves p
  // x-edges among the points up to p, less the first point's own bit
  auto count_x = [](uint64_t s, uint64_t s0) -> uint32_t {
    return (uint32_t)popc(s ^ (s << 1)) - ((uint32_t)s0 & 1u);
  };
  auto next = [&](uint64_t s0, uint64_t sn) -> uint64_t {  // the point after p
    return ((s0 >> 1) | (sn << 63)) << up;
  };
  // the edges leaving p
  const uint64_t ab = A ^ B, ac = A ^ C;
  const uint32_t x = sign(A ^ next(A0, An)) & xin, y = sign(ab), z = sign(ac);
  const uint32_t first = ba + count_x(A, A0) + (uint32_t)popc(ab) + (uint32_t)popc(ac) - y - z;
  // the point before p
  uint64_t Pa = A << 1, Pb = B << 1, Pc = C << 1;
  if (bit == 0) {
    Pa = Pb = Pc = A;
    if (p.q > 0) {
      Pa = b[w - 1];
      Pb = b[w - 1 + sy];
      Pc = b[w - 1 + sz];
    }
  }
  const uint32_t px = sign(Pa ^ A), py = sign(Pa ^ Pb), pz = sign(Pa ^ Pc);
  const uint64_t ya = Y ^ A, yc = Y ^ YC, za = Z ^ A, zb = Z ^ ZB;
  const uint32_t yin = sign(ya), zin = sign(za);  // Y is A in the first row
  bool on[6] = {x != 0u, y != 0u, z != 0u, px != 0u, yin != 0u, zin != 0u};
  const uint32_t id[6] = {
      first, first + x, first + x + y, first - px - py - pz,
      by + count_x(Y, Y0) + (uint32_t)popc(ya) + (uint32_t)popc(yc) - yin - sign(yc) +
          (sign(Y ^ next(Y0, Yn)) & xin),
      bz + count_x(Z, Z0) + (uint32_t)popc(zb) + (uint32_t)popc(za) - zin +
          (sign(Z ^ next(Z0, Zn)) & xin)};
  const f32x4* rec = reinterpret_cast<const f32x4*>(adj);
  f32x4 v[6];
  // unconditional loads (record 0 for an edge that is not there), in flight
  // together
#pragma unroll
  for (int e = 0; e < 6; ++e) {
    on[e] = on[e] && (int64_t)id[e] < n_adj;
    v[e] = n_adj > 0 ? rec[on[e] ? 2 * (int64_t)id[e] + (e < 3 ? 0 : 1) : 0]
                     : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }
  f32x4 acc{0.0f, 0.0f, 0.0f, 0.0f};  // S, G[0..2]
#pragma unroll
  for (int e = 0; e < 6; ++e)
    if (on[e]) acc += v[e];
  return acc;
}

// The sums of a wave's words' endpoints, a lane per endpoint, at their
// slots (1 + the endpoints before; at most two per point).  before: those
// before the words' tile.
template <int WW>
__device__ __forceinline__ void endpoint_sums_wave(const VolGeom& g,
                                                   const uint64_t* __restrict__ b,
                                                   const uint32_t* __restrict__ lpre,
                                                   const Endpoints& ep,
                                                   const VertexAdj* __restrict__ adj,
                                                   const EdgeList& list, f32x4* __restrict__ sums,
                                                   int64_t ww, uint32_t before, uint8_t* mark) {
  const int lane = threadIdx.x & 63;
  const int64_t w = ww + lane;
  const uint64_t e = lane < WW && w < g.nwords ? ep.words[g.word_off + w] : 0ull;
  const uint32_t n = (uint32_t)popc(e);
  if (!__ballot(n != 0u)) return;
  // read when it is needed: most waves of a large volume have left by now
  const int64_t n_adj = edge_count(list), cap = 2 * list.n_points;
  if (n_adj == 0) return;  // the words were not formed
  const uint32_t inc = wave_incl_scan(n), total = wave_last(inc);
  const int64_t slot0 = 1 + (int64_t)before + ep.pre[g.word_off + ww];
  for (uint32_t e0 = 0; e0 < total; e0 += 64u) {  // wave-uniform
    const int wl = item_word(n, inc, e0, mark);
    const uint32_t i = e0 + (uint32_t)lane;
    const uint32_t start = (uint32_t)__shfl((int)(inc - n), wl, 64);
    const uint64_t word = shfl64(e, wl);
    if (i < total && slot0 + i <= cap)
      sums[slot0 + i] = endpoint_sums(g, b, lpre, ep, adj, n_adj, ww + wl,
                                      select_bit(word, (int)(i - start)));
  }
}

// v / h (one-sided) or v / (2 h) along axis d; a power of two divides exactly
// by its reciprocal.
__device__ __forceinline__ float over_step(const VolGeom& g, int d, float v, bool one_sided) {
  if ((g.pow2_h >> d) & 1u) return v * (one_sided ? g.rcp_h[d] : 0.5f * g.rcp_h[d]);
  return v / (one_sided ? g.spacing[d] : 2.0f * g.spacing[d]);
}

// What the point (x, j, k) receives: (S, G) of its own and, along each axis d,
// G[d] of the points before and after it (zero where there is no endpoint).
struct PointTerms {
  f32x4 own;
  float before[3], after[3];
};

// dL/df of the point: f_q in g_q[d] (one-sided stencils on the first and last
// plane), then along each axis f_q = f(p + e_d) for p = q - e_d and
// f_q = f(p - e_d) for p = q + e_d.  INTERIOR: the point is two points or more
// from every border (no one-sided stencil takes part).
template <bool INTERIOR>
__device__ __forceinline__ float combine_point(const VolGeom& g, int x, int j, int k,
                                               const PointTerms& t) {
  float acc = t.own.x;
  if constexpr (INTERIOR) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      acc += over_step(g, d, t.before[d], false);
      acc += -over_step(g, d, t.after[d], false);
    }
    return acc;
  }
  const float G[3] = {t.own.y, t.own.z, t.own.w};
  const int co[3] = {x, j, k};
  const int n[3] = {g.nx, g.ny, g.nz};
  float one = 1.0f;
  asm volatile("" : "+v"(one));  // keeps the quotients in this rare path
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    if (n[d] < 2) continue;
    if (co[d] == 0)
      acc += G[d] * over_step(g, d, -one, true);
    else if (co[d] == n[d] - 1)
      acc += G[d] * over_step(g, d, one, true);
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    if (n[d] < 2) continue;
    if (co[d] >= 1) acc += over_step(g, d, t.before[d], co[d] == 1);
    if (co[d] <= n[d] - 2) acc += -over_step(g, d, t.after[d], co[d] == n[d] - 2);
  }
  return acc;
}

// Zeros over the points of row words [w0, w_end) of a volume: one
// contiguous run of the field (16-byte stores between scalar head and tail).
__device__ __forceinline__ void zero_run(const VolGeom& g, float* __restrict__ out, int64_t w0,
                                         int64_t w_end, int tid, int nt) {
  const WordPos pa = word_pos(g, w0), pb = word_pos(g, w_end - 1);
  const int64_t p0 = (int64_t)pa.q * 64 + (int64_t)g.nx * (pa.j + (int64_t)g.ny * pa.k);
  const int64_t p1 = min((int64_t)pb.q * 64 + 64, (int64_t)g.nx) +
                     (int64_t)g.nx * (pb.j + (int64_t)g.ny * pb.k);
  float* o = out + p0;
  const int64_t n = p1 - p0;
  const int64_t head = min(n, (int64_t)(((16 - (reinterpret_cast<uintptr_t>(o) & 15)) & 15) / 4));
  for (int64_t t = tid; t < head; t += nt) o[t] = 0.0f;
  f32x4* o4 = reinterpret_cast<f32x4*>(o + head);
  const int64_t n4 = (n - head) >> 2;
  for (int64_t t = tid; t < n4; t += nt) o4[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int64_t t = head + 4 * n4 + tid; t < n; t += nt) o[t] = 0.0f;
}

// dL/df of the point (x, j, k) of row word w from the records of its and its
// neighbours' edges, in combine_point's order: an edge list cut below the
// surface's vertices has slots for two endpoints per edge it holds, so that the
// sums of later endpoints have none.
__device__ __forceinline__ float cut_point(const VolGeom& g, const uint64_t* __restrict__ b,
                                           const uint32_t* __restrict__ lpre, const Endpoints& ep,
                                           const VertexAdj* __restrict__ adj, int64_t n_adj,
                                           int64_t w, int x, int j, int k) {
  const int64_t plane = (int64_t)g.wpr * g.ny;
  float acc = 0.0f;
#pragma unroll 1
  for (int n = 0; n < 7; ++n) {  // the point, then before and after it along each axis
    const int d = (n - 1) >> 1, step = n == 0 ? 0 : ((n & 1) ? -1 : 1);
    const int c = d == 0 ? x : (d == 1 ? j : k), size = d == 0 ? g.nx : (d == 1 ? g.ny : g.nz);
    if (n > 0 && (c + step < 0 || c + step >= size)) continue;
    const int xs = n > 0 && d == 0 ? x + step : x;
    const int64_t ws = w + (xs >> 6) - (x >> 6) +
                       (n > 0 && d > 0 ? step * (d == 1 ? (int64_t)g.wpr : plane) : 0);
    const f32x4 v = endpoint_sums(g, b, lpre, ep, adj, n_adj, ws, xs & 63);
    if (n == 0) {
      acc = v.x;
      const float G[3] = {v.y, v.z, v.w};
      const int co[3] = {x, j, k}, nn[3] = {g.nx, g.ny, g.nz};
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        if (co[a] == 0)
          acc += G[a] * over_step(g, a, -1.0f, true);
        else if (co[a] == nn[a] - 1)
          acc += G[a] * over_step(g, a, 1.0f, true);
      }
      continue;
    }
    const float q = d == 0 ? over_step(g, 0, v.y, step < 0 ? x == 1 : x == g.nx - 2)
                           : (d == 1 ? over_step(g, 1, v.z, step < 0 ? j == 1 : j == g.ny - 2)
                                     : over_step(g, 2, v.w, step < 0 ? k == 1 : k == g.nz - 2));
    acc += step < 0 ? q : -q;
  }
  return acc;
}

// What a wave of the gather keeps of its words: the endpoint words of the word
// itself, the rows before and after it and the planes before and after it, the
// slots before their first endpoints, the points that receive something and
// the number of them before the word, the word's first point, and flags:
// bit 0 / 1: the point before / after the word is an endpoint, bit 2: no
// receiving point is within two points of a border.
template <int WW>
struct GatherWave {
  uint64_t ends[5][WW];
  uint64_t recv[WW];
  uint32_t slot[5][WW];
  uint32_t start[WW];
  uint32_t base[WW];
  uint8_t flags[WW];
  uint8_t mark[64];
};

// dL/df of the points of a wave's row words: zeros over all of
// them, then, a lane per point, those that receive something (a wave's stores
// to one address stay in order).  On a surface a row word has about 8 of them
// in 64.  Bound by the lanes' instructions: one shift of an endpoint word puts
// the point's flag in its sign and the endpoints up to the point under a
// popcount, from the neighbours only the one component that the stencil takes
// is read, and waves without points next to a border take a short sum.  Large
// outputs are bound by their zeros (640^3: 162 us of 305 without a surface)
// mixed with the reads.  A lane per point of a word (flags and ranks from
// wave-uniform masks, whole words stored) took 44 us at 256^3 and 334 at
// 640^3 where this takes 23 and 305..317; the points composed in LDS and stored
// once 29 and 323.
template <int WW>
__device__ __forceinline__ void gather_wave(const VolGeom& g, const uint64_t* __restrict__ b,
                                            const uint32_t* __restrict__ lpre, const Endpoints& ep,
                                            const VertexAdj* __restrict__ adj, const EdgeList& list,
                                            const f32x4* __restrict__ sums, uint32_t cap,
                                            float* __restrict__ out, int64_t ww,
                                            GatherWave<WW>& W) {
  const int lane = threadIdx.x & 63;
  const int64_t plane = (int64_t)g.wpr * g.ny;
  const int64_t w = ww + lane;
  uint64_t e[5], r = 0ull;
  int64_t at[5] = {w, w, w, w, w};
  uint32_t flags = 0u, base = 0u;
  if (lane < WW && w < g.nwords && cap != 0u) {
    const WordPos p = word_pos(g, w);
    base = ((uint32_t)p.k * (uint32_t)g.ny + (uint32_t)p.j) * (uint32_t)g.nx + (uint32_t)p.q * 64u;
    const uint64_t* ew = ep.words + g.word_off;
    if (p.j > 0) at[1] = w - g.wpr;
    if (p.has_y) at[2] = w + g.wpr;
    if (p.k > 0) at[3] = w - plane;
    if (p.has_z) at[4] = w + plane;
#pragma unroll
    for (int n = 0; n < 5; ++n) e[n] = ew[at[n]];
    const uint64_t before = ew[p.q > 0 ? w - 1 : w] >> 63;
    const uint64_t after = ew[p.q + 1 < g.wpr ? w + 1 : w];
#pragma unroll
    for (int n = 1; n < 5; ++n)
      if (at[n] == w) e[n] = 0ull;
    flags = (p.q > 0 ? (uint32_t)before : 0u) |
            (p.q + 1 < g.wpr ? ((uint32_t)after & 1u) << 1 : 0u);
    r = e[0] | (e[0] << 1) | (e[0] >> 1) | e[1] | e[2] | e[3] | e[4] | (flags & 1u) |
        ((uint64_t)(flags >> 1) << 63);
    r &= low_mask(g.nx - p.q * 64);
    const uint64_t rim = (p.q == 0 ? 3ull : 0ull) | ~low_mask(g.nx - 2 - p.q * 64);
    if (p.j >= 2 && p.j + 2 < g.ny && p.k >= 2 && p.k + 2 < g.nz && !(r & rim)) flags |= 4u;
  }
  uint32_t tile_first[5], slot[5];
  if (r != 0ull) {  // in flight beside the zeros
#pragma unroll
    for (int n = 0; n < 5; ++n) {
      tile_first[n] = ep.tile[g.tile_off + at[n] / kAdjTile];
      slot[n] = ep.pre[g.word_off + at[n]];
    }
  }
  zero_run(g, out, ww, min(ww + WW, g.nwords), lane, 64);
  if (!__ballot(r != 0ull)) return;
  const int64_t n_adj = edge_count(list);
  if (n_adj == 0) return;  // the words were not formed
  const uint32_t n = (uint32_t)popc(r);
  const uint32_t inc = wave_incl_scan(n), total = wave_last(inc);
  if (r != 0ull) {
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      W.ends[i][lane] = e[i];
      W.slot[i][lane] = tile_first[i] + slot[i];
    }
    W.recv[lane] = r;
    W.start[lane] = inc - n;
    W.base[lane] = base;
    W.flags[lane] = (uint8_t)flags;
  }
  wave_lds_sync();
  const float* sf = reinterpret_cast<const float*>(sums);
  bool cut = false;
  for (uint32_t e0 = 0; e0 < total; e0 += 64u) {  // wave-uniform
    const int i = item_word(n, inc, e0, W.mark);
    const uint32_t t = e0 + (uint32_t)lane;
    if (t >= total) continue;
    const int bit = select_bit(W.recv[i], (int)(t - W.start[i]));
    const int up = 63 - bit;  // brings the point's bit to the sign
    const uint32_t fl = W.flags[i];
    uint32_t slot[7];  // own, then before and after along each axis; slot 0 holds zeros
    {
      const uint64_t own = W.ends[0][i], o = own << up;
      const uint32_t s = W.slot[0][i] + (uint32_t)popc(o);
      const bool on = (int64_t)o < 0;
      const bool before = (int64_t)(((own << 1) | (fl & 1u)) << up) < 0;
      const bool after = (int64_t)(((own >> 1) | ((uint64_t)(fl & 2u) << 62)) << up) < 0;
      slot[0] = on ? s : 0u;
      slot[1] = before ? s - (on ? 1u : 0u) : 0u;
      slot[2] = after ? s + 1u : 0u;
    }
#pragma unroll
    for (int d = 1; d < 3; ++d) {
      const uint64_t b4 = W.ends[2 * d - 1][i] << up, af = W.ends[2 * d][i] << up;
      slot[2 * d + 1] = (int64_t)b4 < 0 ? W.slot[2 * d - 1][i] + (uint32_t)popc(b4) : 0u;
      slot[2 * d + 2] = (int64_t)af < 0 ? W.slot[2 * d][i] + (uint32_t)popc(af) : 0u;
    }
    uint32_t far = slot[0];
#pragma unroll
    for (int q = 1; q < 7; ++q) far = max(far, slot[q]);
    float* o = out + (int64_t)W.base[i] + bit;
    cut = cut || far > cap;  // a cut list: some sums have no slot
#pragma unroll
    for (int q = 0; q < 7; ++q) slot[q] = min(slot[q], cap);
    PointTerms v;
    v.own = sums[slot[0]];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      v.before[d] = sf[4 * (int64_t)slot[2 * d + 1] + 1 + d];
      v.after[d] = sf[4 * (int64_t)slot[2 * d + 2] + 1 + d];
    }
    if (!__ballot(!(fl & 4u))) {
      *o = combine_point<true>(g, 0, 0, 0, v);
    } else {
      const WordPos p = word_pos(g, ww + i);
      *o = combine_point<false>(g, p.q * 64 + bit, p.j, p.k, v);
    }
  }
  if (__builtin_expect(!__ballot(cut), 1)) return;
  for (uint32_t e0 = 0; e0 < total; e0 += 64u) {  // wave-uniform
    const int i = item_word(n, inc, e0, W.mark);
    const uint32_t t = e0 + (uint32_t)lane;
    if (t >= total) continue;
    const int bit = select_bit(W.recv[i], (int)(t - W.start[i]));
    const WordPos p = word_pos(g, ww + i);
    out[(int64_t)W.base[i] + bit] =
        cut_point(g, b, lpre, ep, adj, n_adj, ww + i, p.q * 64 + bit, p.j, p.k);
  }
}

// Widest rows the adjoint takes (nx <= 15872).
constexpr int kMaxGatherWpr = 248;

// Scratch of the adjoint: the vertex records, then the endpoints' sums (slot 0:
// zeros; at most two endpoints per vertex, 16 bytes each).
__host__ __device__ constexpr size_t endpoint_sums_offset(int64_t n_points) {
  return (size_t)(n_points > 0 ? n_points : 0) * sizeof(VertexAdj);
}
__host__ __device__ constexpr size_t adjoint_scratch_bytes(int64_t n_points) {
  return n_points > 0 ? 2 * endpoint_sums_offset(n_points) + 16 : 0;
}
// Words per wave of the sums and the gather of `nwords` row words in `tiles`
// tiles.  Small volumes have too few waves with many words each, and a wave
// goes through its words' points 64 at a time, one round after another; large
// ones have mostly words without points, where a wave of few words is spent on
// finding that out, and fewer lanes have something to do.  Backward in us with
// 8 / 32 / 64 words, Gaussian mixtures of n^3 points: 96 22 / 30 / 41,
// 128 26 / 39 / 53, 160 32 / 32 / 40, 256 73 / 59 / 65, 512 382 / 219 / 221;
// 256 volumes of 32..160 points an axis 668 / 439 / 428; sums + gather of the
// 1024^3 Mandelbulb 2972 / 1754 / 1460, of 64^3 noise 30 / 93 / 177.  Volumes
// of a batch that leave their tiles mostly empty take one wave each (20000 of
// 6 x 7 x 5 points 242 / 83 / 42).
inline int adjoint_wave_words(int64_t nwords, int64_t tiles) {
  if (nwords < 64 * tiles && tiles > 1) return 64;
  return nwords <= (1 << 16) ? 8 : (nwords < (1 << 22) ? 32 : 64);
}
// The last slot (a volume or batch of at most 2^31 points has fewer endpoints).
inline uint32_t last_slot(int64_t n_points) {
  return (uint32_t)std::min<int64_t>(2 * n_points, 0xfffffffe);
}

}  // namespace mc
}  // namespace daxhip
