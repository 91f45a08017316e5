// Isosurfaces of unstructured grids of one cell shape: the reference's
// MarchingTetrahedraCount / MarchingTetrahedraGenerate
// (dax/worklet/MarchingTetrahedra.h:29-143) on UnstructuredGrid<Tetrahedron>
// and MarchingCubesCount / MarchingCubesGenerate (dax/worklet/MarchingCubes.h:
// 53-164) on UnstructuredGrid<Hexahedron>, dispatched through
// DispatcherMapCell and DispatcherGenerateInterpolatedCells
// (dax/cont/DispatcherGenerateInterpolatedCells.h:138-301).
//   count    : per cell the case sum_v (f_v > iso) << v and NumFaces[case]:
//              as a bit per cell and totals per block of cells, or (entries
//              that take them) as a count and an exclusive offset per cell;
//              ids outside the points are reported
//   generate : the triangles' corners in cell order: edge from the table,
//              endpoints ordered by point id, weight (iso - f_A) / (f_B - f_A)
//   dedup    : no grid structure to number edges by: the reference's Sort /
//              Unique / LowerBounds on (EdgeIdFirst, EdgeIdSecond) (:261-301)
//              numbers the distinct pairs in their order; here the pairs are
//              numbered through rows of upper endpoints per lower endpoint,
//              or sorted where those do not fit
//   points   : Lerp(coords[A], coords[B], w) (CompactPointField, :107-141)
#include <algorithm>

#include "algorithms.h"
#include "mc_case_table.h"

namespace daxhip {
namespace ucell {

// Tetrahedra: per case the number of triangles (bits 0-1) and up to 6 edge
// numbers (3 bits each from bit 2) of MarchingTetrahedraTable.h:28-54, in
// the table's order.
__constant__ uint32_t c_tet_cases[16] = {0,      609,    1057, 314246, 1349, 706914,
                                         558250, 1197,   1421, 726026, 476450, 677,
                                         285070, 385,    833,  0};
// Their edges' endpoints (MarchingTetrahedra.h:110-113): kTetEnd0 / kTetEnd1.

// Hexahedra: the marching-cubes case table (packed as in mc_case_table.h)
// (the endpoints of the 12 hexahedron edges, MarchingCubes.h:131-135, are
// kHexEnd0 / kHexEnd1).
__constant__ uint64_t c_hex_cases[256] = DAX_HIP_MC_CASE_TABLE_INIT;

// A case's table entry (its triangle count and edges) and an edge's end
// vertices, packed 4 bits each.
template <int NV>
struct Shape;

constexpr uint64_t pack_ends(const uint8_t (&ends)[12], int n) {
  uint64_t r = 0;
  for (int e = 0; e < n; ++e) r |= (uint64_t)ends[e] << (4 * e);
  return r;
}
constexpr uint8_t kTetEnd0[12] = {0, 1, 2, 3, 3, 3}, kTetEnd1[12] = {1, 2, 0, 0, 1, 2};
constexpr uint8_t kHexEnd0[12] = {0, 1, 3, 0, 4, 5, 7, 4, 0, 1, 2, 3},
                  kHexEnd1[12] = {1, 2, 2, 3, 5, 6, 6, 7, 4, 5, 6, 7};

template <>
struct Shape<4> {
  static constexpr uint64_t kEnd0 = pack_ends(kTetEnd0, 6), kEnd1 = pack_ends(kTetEnd1, 6);
  __device__ static uint64_t entry(int c) { return c_tet_cases[c]; }
  __device__ static int faces(uint64_t t) { return (int)(t & 3u); }
  __device__ static int edge(uint64_t t, int k) { return (int)((t >> (2 + 3 * k)) & 7u); }
};

template <>
struct Shape<8> {
  static constexpr uint64_t kEnd0 = pack_ends(kHexEnd0, 12), kEnd1 = pack_ends(kHexEnd1, 12);
  __device__ static uint64_t entry(int c) { return c_hex_cases[c]; }
  __device__ static int faces(uint64_t t) { return (int)(t >> 60); }
  __device__ static int edge(uint64_t t, int k) { return (int)((t >> (4 * k)) & 15u); }
};
template <int NV>
__device__ __forceinline__ int end0(int e) { return (int)((Shape<NV>::kEnd0 >> (4 * e)) & 15u); }
template <int NV>
__device__ __forceinline__ int end1(int e) { return (int)((Shape<NV>::kEnd1 >> (4 * e)) & 15u); }

// The NV point ids of cell t; with kVec the rows are read as 16-byte loads
// (the connectivity is 16-byte aligned).
template <int NV, bool kVec>
__device__ __forceinline__ void load_ids(const int32_t* __restrict__ cells, int64_t t, int* id) {
  if (kVec) {
    const int4* p = (const int4*)(cells + NV * t);
#pragma unroll
    for (int q = 0; q < NV / 4; ++q) {
      const int4 v = p[q];
      id[4 * q + 0] = v.x;
      id[4 * q + 1] = v.y;
      id[4 * q + 2] = v.z;
      id[4 * q + 3] = v.w;
    }
  } else {
#pragma unroll
    for (int v = 0; v < NV; ++v) id[v] = cells[NV * t + v];
  }
}

template <int NV, bool kVec>
__global__ __launch_bounds__(256) void k_count(const int32_t* __restrict__ cells, int64_t n_cells,
                                               const float* __restrict__ field, int64_t n_points,
                                               float iso, int32_t* __restrict__ counts,
                                               int32_t* __restrict__ bad) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_cells) return;
  int id[NV];
  load_ids<NV, kVec>(cells, t, id);
  bool ok = true;
#pragma unroll
  for (int v = 0; v < NV; ++v) ok = ok && id[v] >= 0 && id[v] < n_points;
  if (!ok) {
    counts[t] = 0;
    *bad = 1;
    return;
  }
  int c = 0;
#pragma unroll
  for (int v = 0; v < NV; ++v) c |= (field[id[v]] > iso) << v;
  counts[t] = Shape<NV>::faces(Shape<NV>::entry(c));
}

__device__ __forceinline__ void lerp3(const float* __restrict__ pts, int64_t a, int64_t b, float w,
                                      float* out) {
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const float pa = pts[3 * a + d], pb = pts[3 * b + d];
    out[d] = pa + w * (pb - pa);
  }
}

// Notes the corner edge (a, b), a < b: the pair, and a byte at a.  The bytes
// become bits in k_point_prefix: plain stores, where atomicOr on the words
// themselves crosses the XCDs' L2s (2.06 M corners: generate 74 us, 25
// with bytes).
__device__ __forceinline__ void note_edge(int2* __restrict__ pairs, uint8_t* __restrict__ used,
                                          int64_t i, int a, int b) {
  pairs[i] = make_int2(a, b);
  if (used) used[a] = 1;  // null: the edges are sorted
}

// Corners of every triangle: with pairs, each corner's edge (dedup); without,
// the corner's point record, coordinates and identity connectivity.
//
// A thread per output triangle (the reference's UpperBounds and visit index,
// DispatcherGenerateInterpolatedCells.h:196-212): its cell is the last one
// whose exclusive offset is <= the triangle, its visit index the difference.
template <int NV, bool kVec>
__global__ __launch_bounds__(256) void k_generate(
    const int32_t* __restrict__ cells, int64_t n_cells, const float* __restrict__ field,
    const float* __restrict__ pts, int64_t n_points, float iso, int64_t n_tris,
    const int32_t* __restrict__ offs, int2* __restrict__ pairs, uint8_t* __restrict__ used,
    int32_t* __restrict__ first,
    int32_t* __restrict__ second, float* __restrict__ weight, float* __restrict__ verts,
    int32_t* __restrict__ conn) {
  const int64_t tri = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (tri >= n_tris) return;
  int64_t lo = 0, hi = n_cells;  // offs[0] = 0 <= tri
  while (hi - lo > 1) {
    const int64_t mid = (lo + hi) >> 1;
    if ((int64_t)offs[mid] <= tri)
      lo = mid;
    else
      hi = mid;
  }
  const int64_t t = lo;
  const int visit = (int)(tri - offs[t]);
  int id[NV];
  load_ids<NV, kVec>(cells, t, id);
  float f[NV];
  int c = 0;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    f[v] = field[id[v]];
    c |= (f[v] > iso) << v;
  }
  const uint64_t entry = Shape<NV>::entry(c);
  if (visit >= Shape<NV>::faces(entry)) {  // offsets not from this field's counts
    if (pairs)
      for (int k = 0; k < 3; ++k) pairs[3 * tri + k] = make_int2(-1, -1);  // no edge
    return;
  }
  const int64_t base = 3 * (int64_t)offs[t];
  for (int k = 3 * visit; k < 3 * visit + 3; ++k) {
    const int e = Shape<NV>::edge(entry, k);
    int va = end0<NV>(e), vb = end1<NV>(e);
    int ia = 0, ib = 0;
    float fa = 0.0f, fb = 0.0f;
    // registers indexed by a run-time vertex: select instead of a local array
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      if (v == va) {
        ia = id[v];
        fa = f[v];
      }
      if (v == vb) {
        ib = id[v];
        fb = f[v];
      }
    }
    if (!(ia < ib)) {  // endpoints ordered by point id (ties keep the swap)
      const int si = ia;
      ia = ib;
      ib = si;
      const float sf = fa;
      fa = fb;
      fb = sf;
    }
    const int64_t i = base + k;
    if (pairs) {
      note_edge(pairs, used, i, ia, ib);
    } else {
      const float w = (iso - fa) / (fb - fa);
      first[i] = ia;
      second[i] = ib;
      weight[i] = w;
      float xyz[3];
      lerp3(pts, ia, ib, w, xyz);
      verts[3 * i + 0] = xyz[0];
      verts[3 * i + 1] = xyz[1];
      verts[3 * i + 2] = xyz[2];
      conn[i] = (int32_t)i;
    }
  }
}

// {triangle total, bad-id flag} for one read-back: the last offset plus the
// last count.
__global__ void k_count_result(const int32_t* __restrict__ offs,
                               const int32_t* __restrict__ counts, int64_t n,
                               const int32_t* __restrict__ bad, int32_t* __restrict__ out2) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    out2[0] = offs[n - 1] + counts[n - 1];
    out2[1] = *bad;
  }
}

// 1 where a sorted key starts a run of equal keys.
__global__ __launch_bounds__(256) void k_run_starts(const uint64_t* __restrict__ sorted,
                                                    int64_t n, int32_t* __restrict__ flag) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) flag[i] = (i == 0 || sorted[i] != sorted[i - 1]) ? 1 : 0;
}

// Each corner's point (the reference's LowerBounds of its key in the unique
// keys): sorted position i holds corner idx[i], whose point is the number of
// its run, i.e. the run starts up to and including i, less one; `rank` is
// the exclusive scan of the run starts, so a position inside a run (not a
// start) subtracts one.
__global__ __launch_bounds__(256) void k_corner_points(const uint64_t* __restrict__ sorted,
                                                       const int32_t* __restrict__ idx,
                                                       const int32_t* __restrict__ rank, int64_t n,
                                                       int32_t* __restrict__ conn) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const bool start = i == 0 || sorted[i] != sorted[i - 1];
  const int32_t c = idx[i];
  if (c >= 0 && c < n) conn[c] = rank[i] - (start ? 0 : 1);  // always in range: a permutation
}

// The unique points (sorted keys): records, weights and coordinates.
__global__ __launch_bounds__(256) void k_points(const uint64_t* __restrict__ sorted,
                                                const int32_t* __restrict__ rank, int64_t n,
                                                uint64_t n_points, const float* __restrict__ field,
                                                const float* __restrict__ pts, float iso,
                                                int32_t* __restrict__ first,
                                                int32_t* __restrict__ second,
                                                float* __restrict__ weight,
                                                float* __restrict__ verts) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || (i > 0 && sorted[i] == sorted[i - 1])) return;  // a run's first key only
  const int64_t u = rank[i];
  const uint64_t key = sorted[i];
  const int32_t a = (int32_t)(key / n_points), b = (int32_t)(key - (uint64_t)a * n_points);
  const float fa = field[a], fb = field[b];
  const float w = (iso - fa) / (fb - fa);
  if (first) first[u] = a;
  if (second) second[u] = b;
  if (weight) weight[u] = w;
  float xyz[3];
  lerp3(pts, a, b, w, xyz);
  verts[3 * u + 0] = xyz[0];
  verts[3 * u + 1] = xyz[1];
  verts[3 * u + 2] = xyz[2];
}

// ---- count and generate by blocks of cells ---------------------------------
// count: a block of 256 threads takes kCellBlock cells and writes a bit per
// cell with triangles and the block's triangle total (bit 31: a cell with an
// id outside the points); one block scans the totals.  generate: a wave takes
// a block's cells with triangles, 64 at a time, as the uniform grid's generate
// does: words of bits mark their first cell's lane, a prefix maximum finds
// each lane's word, a wave scan of the triangle counts places the triangles.
// Against a count and an offset per cell (written, scanned, and searched by
// every triangle) the cells' ids are all that is read in full: 12.3 M
// tetrahedra 105 + 14 us -> 62 + 11, 16.6 M hexahedra 166 + 41 -> 125 + 25.
constexpr int kCellBlock = 1024;
constexpr int kCellWords = kCellBlock / 64;
constexpr uint32_t kBadCells = 0x80000000u;

template <int NV, bool kVec>
__global__ __launch_bounds__(256) void k_count_blocks(const int32_t* __restrict__ cells,
                                                      int64_t n_cells,
                                                      const float* __restrict__ field,
                                                      int64_t n_points, float iso,
                                                      uint64_t* __restrict__ bits,
                                                      uint32_t* __restrict__ sums) {
  constexpr int kPer = kCellBlock / 256;
  __shared__ uint8_t s_faces[1 << NV];
  __shared__ uint32_t s_sum[4];
  if (threadIdx.x < (1 << NV))
    s_faces[threadIdx.x] = (uint8_t)Shape<NV>::faces(Shape<NV>::entry((int)threadIdx.x));
  __syncthreads();
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int64_t c0 = (int64_t)blockIdx.x * kCellBlock + wv * (kPer * 64) + lane;
  int id[kPer][NV];
  bool ok[kPer];
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int64_t c = c0 + 64 * u;
    ok[u] = c < n_cells;
#pragma unroll
    for (int v = 0; v < NV; ++v) id[u][v] = 0;
    if (ok[u]) load_ids<NV, kVec>(cells, c, id[u]);
  }
  bool bad = false;
  uint32_t total = 0u;
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    bool in = ok[u];
#pragma unroll
    for (int v = 0; v < NV; ++v) in = in && id[u][v] >= 0 && id[u][v] < n_points;
    bad = bad || (ok[u] && !in);
    int cs = 0;
    if (in) {
#pragma unroll
      for (int v = 0; v < NV; ++v) cs |= (field[id[u][v]] > iso) << v;
    }
    const uint32_t nf = in ? (uint32_t)s_faces[cs] : 0u;
    const uint64_t active = __ballot(nf != 0u);
    const int64_t w = (int64_t)blockIdx.x * kCellWords + wv * kPer + u;
    if (lane == 0) bits[w] = active;
    total += wave_sum(nf);
  }
  const bool any_bad = __ballot(bad) != 0ull;
  if (lane == 0) s_sum[wv] = total | (any_bad ? kBadCells : 0u);
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t t = 0u, flag = 0u;
    for (int q = 0; q < 4; ++q) {
      t += s_sum[q] & ~kBadCells;
      flag |= s_sum[q] & kBadCells;
    }
    sums[blockIdx.x] = t | flag;
  }
}

// Exclusive scan in place of n values (n_dev, when given, counts rows: their
// tiles bound n) by one block; the total and the OR of the
// values' top bits go to out2 and, with `host`, to pinned memory, and a flag
// with them.
constexpr int kScanBlock = 1024;
constexpr int kRowTile = 64;  // rows per tile of the dedup, below
__global__ __launch_bounds__(kScanBlock) void k_scan_block(uint32_t* __restrict__ v, int64_t n,
                                                           const uint32_t* __restrict__ n_dev,
                                                           uint32_t* __restrict__ out2,
                                                           const uint32_t* __restrict__ flag,
                                                           int64_t* __restrict__ host) {
  __shared__ uint32_t s_scan[kScanBlock / 64];
  if (n_dev) n = min(n, ceil_div((int64_t)*n_dev, (int64_t)kRowTile));
  unsigned long long carry = 0ull;
  bool top = false;
  for (int64_t c0 = 0; c0 < n; c0 += kScanBlock * kScanChunk) {
    const int64_t i0 = c0 + (int64_t)threadIdx.x * kScanChunk;
    u32x4 x[kScanChunk / 4];
    load_chunk(v, i0, n, x);
    uint32_t sum = 0u, bits = 0u, total;
#pragma unroll
    for (int q = 0; q < kScanChunk; ++q) {
      bits |= x[q / 4][q % 4];
      x[q / 4][q % 4] &= ~kBadCells;
      sum += x[q / 4][q % 4];
    }
    top = top || (bits & kBadCells);
    const uint32_t run = (uint32_t)carry + block_excl_scan(sum, total, s_scan);
    carry += total;
    store_prefixes(v, i0, n, x, run);
  }
  const bool any_top = __syncthreads_or(top);
  if (threadIdx.x == 0) {
    if (out2) {
      out2[0] = (uint32_t)min(carry, 0xffffffffull);
      out2[1] = any_top ? 1u : 0u;
    }
    if (host) {
      __hip_atomic_store(host, (int64_t)carry, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      __hip_atomic_store(host + 1, (int64_t)(any_top || (flag && *flag)), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

// What a wave of the generate keeps of a round of 64 cells.
template <int NV>
struct CellWave {
  uint64_t entry[64];
  int32_t id[NV][64];
  float f[NV][64];
  uint16_t first[64];
  uint8_t tri_cell[5 * 64];
  uint8_t word_mark[64];
};

template <int NV, bool kVec, bool kDedup>
__global__ __launch_bounds__(256) void k_generate_blocks(
    const int32_t* __restrict__ cells, int64_t n_blocks, const float* __restrict__ field,
    const float* __restrict__ pts, float iso, int64_t n_tris, const uint64_t* __restrict__ bits,
    const uint32_t* __restrict__ sums, int2* __restrict__ pairs, uint8_t* __restrict__ used,
    int32_t* __restrict__ first, int32_t* __restrict__ second, float* __restrict__ weight,
    float* __restrict__ verts, int32_t* __restrict__ conn) {
  __shared__ CellWave<NV> s_wave[4];
  CellWave<NV>& W = s_wave[threadIdx.x >> 6];
  const int lane = threadIdx.x & 63;
  const int64_t blk = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (blk >= n_blocks) return;  // whole waves; no block barrier follows
  const uint64_t act = lane < kCellWords ? bits[blk * kCellWords + lane] : 0ull;
  const uint32_t nc = (uint32_t)__popcll(act);
  const uint32_t inc = wave_incl_scan(nc), n_act = wave_last(inc), start = inc - nc;
  int64_t tri = n_act ? (int64_t)sums[blk] : 0;
  for (uint32_t r0 = 0; r0 < n_act; r0 += 64u) {  // wave-uniform
    W.word_mark[lane] = 0;
    wave_lds_sync();
    if (nc != 0u && start < r0 + 64u && inc > r0)
      W.word_mark[max(start, r0) - r0] = (uint8_t)(lane + 1);
    wave_lds_sync();
    const int wl = (int)wave_incl_max((uint32_t)W.word_mark[lane]) - 1;
    const uint32_t slot = r0 + (uint32_t)lane;
    const bool valid = slot < n_act;
    const uint32_t wstart = (uint32_t)__shfl((int)start, wl, 64);
    const uint64_t word = ((uint64_t)(uint32_t)__shfl((int)(uint32_t)(act >> 32), wl, 64) << 32) |
                          (uint32_t)__shfl((int)(uint32_t)act, wl, 64);
    const int bit = select_bit(word, valid ? (int)(slot - wstart) : 0);
    // an invalid lane repeats its word's first cell, which has triangles
    const int64_t c = blk * kCellBlock + 64 * wl + bit;
    int id[NV];
    load_ids<NV, kVec>(cells, c, id);
    float f[NV];
    int cs = 0;
#pragma unroll
    for (int v = 0; v < NV; ++v) f[v] = field[id[v]];  // ids checked by the count
#pragma unroll
    for (int v = 0; v < NV; ++v) cs |= (f[v] > iso) << v;
    const uint64_t entry = Shape<NV>::entry(cs);
    const uint32_t nf = valid ? (uint32_t)Shape<NV>::faces(entry) : 0u;
    const uint32_t finc = wave_incl_scan(nf), n_round = wave_last(finc), ffirst = finc - nf;
    W.entry[lane] = entry;
    W.first[lane] = (uint16_t)ffirst;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      W.id[v][lane] = id[v];
      if (!kDedup) W.f[v][lane] = f[v];
    }
#pragma unroll
    for (uint32_t t = 0; t < 5u; ++t)
      if (t < nf) W.tri_cell[ffirst + t] = (uint8_t)lane;
    wave_lds_sync();
    for (uint32_t tl = (uint32_t)lane; tl < n_round; tl += 64u) {
      const int cl = (int)W.tri_cell[tl];
      const int visit = (int)(tl - W.first[cl]);
      const uint64_t en = W.entry[cl];
      const int64_t t = tri + tl;
      if (t >= n_tris) continue;  // a field changed since the count
#pragma unroll
      for (int v = 0; v < 3; ++v) {
        const int e = Shape<NV>::edge(en, 3 * visit + v);
        const int va = end0<NV>(e), vb = end1<NV>(e);
        const int ia = W.id[va][cl], ib = W.id[vb][cl];
        const bool swap = !(ia < ib);  // endpoints ordered by point id
        const int a = swap ? ib : ia, b = swap ? ia : ib;
        const int64_t i = 3 * t + v;
        if (kDedup) {
          note_edge(pairs, used, i, a, b);
        } else {
          const float fva = W.f[va][cl], fvb = W.f[vb][cl];
          const float fa = swap ? fvb : fva, fb = swap ? fva : fvb;
          const float w = (iso - fa) / (fb - fa);
          first[i] = a;
          second[i] = b;
          weight[i] = w;
          float xyz[3];
          lerp3(pts, a, b, w, xyz);
          verts[3 * i + 0] = xyz[0];
          verts[3 * i + 1] = xyz[1];
          verts[3 * i + 2] = xyz[2];
          conn[i] = (int32_t)i;
        }
      }
    }
    tri += n_round;
    wave_lds_sync();  // the round's LDS is reused
  }
}

// ---- dedup -------------------------------------------------------------------
// The corners' edges (A, B) numbered in the order of their pairs without
// sorting them all: the lower endpoints A are ranked by the words of their bits;
// the corners are listed by tile of kRowTile ranks (a block reserves room for
// the few tiles its corners fall into), and a block per tile finds its distinct
// pairs in an LDS table, places them by rank and upper endpoint, and numbers its
// corners within the tile; a scan of the tiles' sizes makes the numbers final.
// Any order of insertion gives the same numbers.  A tile of more pairs than the
// table takes goes through its ranks in parts.  A lower endpoint with more
// active edges up from it than that, or a tile of very many corners, sets a flag
// and the general sort is run instead.
//
// The sort's six radix passes and the scans around them took 220 us for 540 K
// corners and 370 for 2.06 M; rows in global memory 62 and 133 us for the
// insertion alone (atomics across the XCDs' L2s); this chain takes 42 and 99 us,
// besides three scans of 4.  Rows of at most 16 edges in LDS instead of the table
// took 18 us for what now takes 17 (42 and 38), but sent every mesh with a longer
// row to the sort: three million unshared tetrahedra 1681 us, now 793.
constexpr int kPointTile = 256;

// 64 points' bits and their exclusive popcount prefix within a tile of
// kPointTile words (one 16-byte load ranks a point).
struct alignas(16) PointWord {
  unsigned long long bits;
  uint32_t pre, pad;
};

struct DedupState {
  uint32_t rows;      // lower endpoints
  uint32_t rows_top;  // (k_scan_block's second word)
  uint32_t overflow;  // to be sorted
  uint32_t pad;
};

// A corner in its tile's list.
struct TileCorner {
  int32_t corner, b;
  uint32_t row;  // within the tile
};

__global__ __launch_bounds__(256) void k_clear16(uint4* __restrict__ p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = make_uint4(0u, 0u, 0u, 0u);
}

// Bits and prefixes of the noted points: a thread per word gathers its 64
// bytes (0 or 1 each; the bytes run to whole words).
__global__ __launch_bounds__(kPointTile) void k_point_prefix(const uint8_t* __restrict__ used,
                                                             PointWord* __restrict__ pw,
                                                             int64_t n,
                                                             uint32_t* __restrict__ tile) {
  __shared__ uint32_t s_scan[kPointTile / 64];
  const int64_t w = (int64_t)blockIdx.x * kPointTile + threadIdx.x;
  uint64_t bits = 0ull;
  if (w < n) {
    const uint4* p = reinterpret_cast<const uint4*>(used + 64 * w);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint4 v = p[q];
      const uint32_t x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int d = 0; d < 4; ++d)  // bytes 0/1 at bits 0, 8, 16, 24 to bits 0..3
        bits |= (uint64_t)((x[d] * 0x01020408u) >> 24 & 15u) << (16 * q + 4 * d);
    }
  }
  uint32_t total;
  const uint32_t pre = block_excl_scan((uint32_t)__popcll(bits), total, s_scan);
  if (w < n)
    *reinterpret_cast<uint4*>(pw + w) =
        make_uint4((uint32_t)bits, (uint32_t)(bits >> 32), pre, 0u);
  if (threadIdx.x == 0) tile[blockIdx.x] = total;
}

__device__ __forceinline__ uint32_t point_rank(const PointWord* __restrict__ pw,
                                               const uint32_t* __restrict__ tile, int a) {
  const uint4 q = *reinterpret_cast<const uint4*>(pw + (a >> 6));
  const uint64_t below = (((uint64_t)q.y << 32) | q.x) & ((1ull << (a & 63)) - 1ull);
  return tile[(a >> 6) / kPointTile] + q.z + (uint32_t)__popcll(below);
}

// A corner whose field changed after the count may hold no edge: it is left
// out of the points and gets number 0.
__device__ __forceinline__ bool is_edge(int2 e, int64_t n_points) {
  return (int64_t)(uint32_t)e.x < n_points && (int64_t)(uint32_t)e.y < n_points;
}

constexpr uint32_t kNoRow = 0xffffffffu;

// Row of every corner and its place among its tile's corners.  A block takes
// kListCorners corners and counts them by tile in an LDS table (open
// addressing, twice as many entries as there can be tiles), so that one global
// atomic per block and tile reserves their places: with one per wave and tile
// the launch took 52 us for 540 K corners and 94 for 2.06 M (neighbouring
// waves wait for the same counters), now 10 and 25.
// A tile has some 700 corners (2.06 M in 2900 tiles); beyond kMaxTileCorners
// going through its ranks in parts costs more than the sort.
constexpr int kListCorners = 1024;
constexpr uint32_t kMaxTileCorners = 1 << 14;
__global__ __launch_bounds__(256) void k_corner_rows(const int2* __restrict__ pairs, int64_t n,
                                                     int64_t n_points,
                                                     const PointWord* __restrict__ pw,
                                                     const uint32_t* __restrict__ ptile,
                                                     uint32_t* __restrict__ count,
                                                     uint2* __restrict__ row_place,
                                                     DedupState* __restrict__ st) {
  constexpr int kPer = kListCorners / 256;
  constexpr uint32_t kTable = 2 * kListCorners;
  __shared__ uint32_t s_key[kTable], s_cnt[kTable];
  for (uint32_t h = threadIdx.x; h < kTable; h += 256u) {
    s_key[h] = kNoRow;
    s_cnt[h] = 0u;
  }
  const uint32_t rows = st->rows;
  uint32_t r[kPer], slot[kPer], place[kPer];
  const int64_t i0 = (int64_t)blockIdx.x * kListCorners + threadIdx.x;
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int64_t i = i0 + 256 * u;
    r[u] = kNoRow;
    if (i < n) {
      const int2 e = pairs[i];
      if (is_edge(e, n_points)) r[u] = point_rank(pw, ptile, e.x);
      if (r[u] >= rows) r[u] = kNoRow;
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    slot[u] = place[u] = 0u;
    if (r[u] == kNoRow) continue;
    const uint32_t t = r[u] / kRowTile;
    uint32_t h = (t * 2654435761u) & (kTable - 1u);
    while (true) {  // at most kListCorners keys in twice as many entries
      const uint32_t have = atomicCAS(&s_key[h], kNoRow, t);
      if (have == kNoRow || have == t) break;
      h = (h + 1u) & (kTable - 1u);
    }
    slot[u] = h;
    place[u] = atomicAdd(&s_cnt[h], 1u);
  }
  __syncthreads();
  for (uint32_t h = threadIdx.x; h < kTable; h += 256u)
    if (s_cnt[h]) {
      const uint32_t first = atomicAdd(&count[s_key[h]], s_cnt[h]);
      if (first + s_cnt[h] > kMaxTileCorners) st->overflow = 1u;
      s_cnt[h] = first;  // the first place
    }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int64_t i = i0 + 256 * u;
    if (i < n) row_place[i] = make_uint2(r[u], place[u] + s_cnt[slot[u]]);
  }
}

// The corners into their tiles' lists (start: the tiles' first entries).
__global__ __launch_bounds__(256) void k_list_corners(const int2* __restrict__ pairs, int64_t n,
                                                      const uint2* __restrict__ row_place,
                                                      const uint32_t* __restrict__ start,
                                                      const DedupState* __restrict__ st,
                                                      TileCorner* __restrict__ list) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || st->overflow) return;
  const uint2 rp = row_place[i];
  if (rp.x == kNoRow) return;
  const int64_t at = (int64_t)start[rp.x / kRowTile] + rp.y;
  if (at >= n) return;  // always below: the places are the counts'
  const TileCorner c{(int32_t)i, pairs[i].y, rp.x % kRowTile};
  __builtin_memcpy(&list[at], &c, sizeof(c));
}

// A block per tile of rows (the grid loops: their number is the device's).
// Leaves every corner's number within its tile in place[corner].y and the tile's
// distinct edges, in the order of their numbers, from its first corner's place in
// the list on (it has no more edges than corners).  64 rows per tile: with 256
// the 120 tiles of the 128^3 tetrahedra's surface left half the CUs idle (27 us,
// now 12.4).  Bound by the chain of loads and barriers of a tile: a thread has its
// four corners' loads in flight together, and what follows the table runs over the
// distinct edges.  512 of them: at 1024 fewer tiles are taken in two passes, but
// fewer blocks fit a CU (256^3 hexahedra 28.4 us, now 24.1; three million unshared
// tetrahedra 887 us in all, now 793; 40 fans of 5000 271, now 313).
constexpr uint32_t kTileEdges = 512;  // distinct edges of a pass over the tile, at most
constexpr uint32_t kTileTable = 2 * kTileEdges;
constexpr int kTilePer = 4;           // corners per thread and turn
__global__ __launch_bounds__(256) void k_tile_edges(
    const int2* __restrict__ pairs, const TileCorner* __restrict__ list,
    const uint32_t* __restrict__ start, const uint32_t* __restrict__ n_list,
    int2* __restrict__ edges, uint32_t* __restrict__ sizes, DedupState* __restrict__ st,
    uint2* __restrict__ place) {
  __shared__ unsigned long long s_key[kTileTable];  // (row + 1) << 32 | upper endpoint; 0: free
  __shared__ uint32_t s_at[kTileTable];        // an entry's corner, then its number
  __shared__ uint16_t s_entry[kTileEdges + 256], s_pos[kTileEdges + 256];  // by order of arrival
  __shared__ uint32_t s_b[kTileEdges];         // upper endpoints by row
  __shared__ uint32_t s_cnt[kRowTile], s_first[kRowTile];
  __shared__ uint32_t s_edges, s_stop;
  const uint32_t tid = threadIdx.x;
  const int64_t n_tiles = ceil_div((int64_t)st->rows, (int64_t)kRowTile);
  for (int64_t t = blockIdx.x; t < n_tiles; t += gridDim.x) {
    if (tid == 0) s_stop = __hip_atomic_load(&st->overflow, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t c0 = start[t], c1 = t + 1 < n_tiles ? start[t + 1] : *n_list;
    uint32_t total = 0u, r0 = 0u, span = kRowTile;
    TileCorner e[kTilePer];
    uint32_t at[kTilePer];
    auto key_of = [](const TileCorner& c) -> unsigned long long {
      return ((unsigned long long)(c.row + 1u) << 32) | (uint32_t)c.b;
    };
    auto load = [&](uint32_t base) {  // rows outside the pass: none
#pragma unroll
      for (int u = 0; u < kTilePer; ++u) {
        const uint32_t c = base + 256u * u + tid;
        e[u].row = kNoRow;
        if (c < c1) __builtin_memcpy(&e[u], &list[c], sizeof(e[u]));
      }
    };
    // the key's entry, or the free one that ends its chain (never more than
    // kTileEdges + 256 keys in the table)
    auto find = [&](const TileCorner& c) -> uint32_t {
      uint32_t h = ((uint32_t)c.b * 2654435761u + c.row * 0x9e3779b9u) >> 12;
      while (true) {
        h &= kTileTable - 1u;
        const unsigned long long have =
            __hip_atomic_load(&s_key[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (have == 0ull || have == key_of(c)) return h;
        ++h;
      }
    };
    while (r0 < (uint32_t)kRowTile) {
      for (uint32_t h = tid; h < kTileTable; h += 256u) s_key[h] = 0ull;
      if (tid < kRowTile) s_cnt[tid] = 0u;
      if (tid == 0) s_edges = 0u;
      __syncthreads();
      if (s_stop) return;  // uniform: written before the first pass
      for (uint32_t base = c0; base < c1; base += 256u * kTilePer) {
        load(base);
#pragma unroll
        for (int u = 0; u < kTilePer; ++u) {
          at[u] = 0u;
          if (e[u].row - r0 >= span) continue;
          if (__hip_atomic_load(&s_edges, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) >
              kTileEdges)
            continue;
          while (true) {
            const uint32_t h = find(e[u]);
            const unsigned long long have = atomicCAS(&s_key[h], 0ull, key_of(e[u]));
            if (have == 0ull) {  // one winner
              const uint32_t i = atomicAdd(&s_edges, 1u);
              s_entry[i] = (uint16_t)h;
              s_at[h] = (uint32_t)e[u].corner;
              s_pos[i] = (uint16_t)atomicAdd(&s_cnt[e[u].row], 1u);
            }
            at[u] = h;
            if (have == 0ull || have == key_of(e[u])) break;
          }
        }
      }
      __syncthreads();
      const uint32_t n = s_edges;
      if (n > kTileEdges) {  // uniform
        __syncthreads();
        if (span == 1u) {
          if (tid == 0) st->overflow = 1u;
          return;
        }
        span /= 2u;
        continue;
      }
      if (tid < kRowTile) {  // wave 0: the rows' first numbers
        const uint32_t cnt = s_cnt[tid];
        s_first[tid] = wave_incl_scan(cnt) - cnt;
      }
      __syncthreads();
      for (uint32_t i = tid; i < n; i += 256u) {
        const unsigned long long key = s_key[s_entry[i]];
        s_b[s_first[(uint32_t)(key >> 32) - 1u] + s_pos[i]] = (uint32_t)key;
      }
      __syncthreads();
      for (uint32_t i = tid; i < n; i += 256u) {
        const uint32_t h = s_entry[i];
        const uint32_t row = (uint32_t)(s_key[h] >> 32) - 1u, b = (uint32_t)s_key[h];
        const int a = pairs[s_at[h]].x;
        uint32_t k = s_first[row];
        for (uint32_t q = 0; q < s_cnt[row]; ++q) k += s_b[s_first[row] + q] < b;
        edges[c0 + total + k] = make_int2(a, (int)b);
        s_at[h] = k;
      }
      __syncthreads();
      const bool kept = c1 - c0 <= 256u * kTilePer;  // the corners are still in registers
      for (uint32_t base = c0; base < c1; base += 256u * kTilePer) {
        if (!kept) load(base);
#pragma unroll
        for (int u = 0; u < kTilePer; ++u)
          if (e[u].row - r0 < span)
            place[e[u].corner].y = total + s_at[kept ? at[u] : find(e[u])];
      }
      total += n;
      r0 += span;
      __syncthreads();  // LDS reused
    }
    if (tid == 0) sizes[t] = total;
  }
}

// The unique points, a block per tile: records, weights and coordinates.
__global__ __launch_bounds__(256) void k_tile_points(
    const int2* __restrict__ edges, const uint32_t* __restrict__ start,
    const uint32_t* __restrict__ n_list, const DedupState* __restrict__ st,
    const uint32_t* __restrict__ tile, const uint32_t* __restrict__ n_edges, int64_t max_points,
    const float* __restrict__ field, const float* __restrict__ pts, float iso,
    int32_t* __restrict__ first, int32_t* __restrict__ second, float* __restrict__ weight,
    float* __restrict__ verts) {
  if (st->overflow) return;
  const int lane = threadIdx.x;
  const int64_t n_tiles = ceil_div((int64_t)st->rows, (int64_t)kRowTile);
  const int64_t step = gridDim.x;
  for (int64_t t = blockIdx.x; t < n_tiles; t += step) {
    const uint32_t u0 = tile[t], u1 = t + 1 < n_tiles ? tile[t + 1] : *n_edges;
    const int2* e0 = edges + start[t];
    for (int64_t u = (int64_t)u0 + lane; u < u1 && u < max_points; u += 256) {
      const int2 e = e0[u - u0];
      const float fa = field[e.x];
      const float w = (iso - fa) / (field[e.y] - fa);
      if (first) first[u] = e.x;
      if (second) second[u] = e.y;
      if (weight) weight[u] = w;
      float xyz[3];
      lerp3(pts, e.x, e.y, w, xyz);
      __builtin_memcpy(verts + 3 * u, xyz, 12);
    }
  }
}

// The corners' numbers within their tiles made final.
__global__ __launch_bounds__(256) void k_number_corners(int64_t n,
                                                        const DedupState* __restrict__ st,
                                                        const uint32_t* __restrict__ tile,
                                                        const uint2* __restrict__ place,
                                                        int32_t* __restrict__ conn) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || st->overflow) return;
  const uint2 p = place[i];
  conn[i] = p.x == kNoRow ? 0 : (int32_t)(tile[p.x / kRowTile] + p.y);
}

// The general path's sort keys A * P + B and their corner indices, from the
// pairs (in place: a thread rewrites its own).
__global__ __launch_bounds__(256) void k_pair_keys(uint64_t* __restrict__ keys, int64_t n,
                                                   uint64_t n_points, int32_t* __restrict__ idx) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int2 e = ((const int2*)keys)[i];
  // (a corner without an edge stands as point 0 twice)
  keys[i] = is_edge(e, (int64_t)n_points)
                ? (uint64_t)(uint32_t)e.x * n_points + (uint64_t)(uint32_t)e.y
                : 0ull;
  idx[i] = (int32_t)i;
}

inline bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

template <int NV>
int count_cells(const char* name, const int32_t* d_cells, int64_t n_cells, const float* d_field,
                int64_t n_points, float iso, int32_t* d_counts, int32_t* d_offsets,
                int64_t* h_tris, void* stream) {
  if (n_cells < 0 || n_points < 0 || n_points > 0x7fffffffLL || !h_tris ||
      n_cells > 0x7fffffffLL / NV ||
      (n_cells > 0 && (!d_cells || !d_field || !d_counts || !d_offsets))) {
    set_error("%s: bad arguments", name);
    return DAX_HIP_BAD_VALUE;
  }
  *h_tris = 0;
  if (n_cells == 0) return DAX_HIP_OK;
  hipStream_t s = (hipStream_t)stream;
  TempBuf flag(s);  // set when a cell references a point outside [0, n_points)
  int rc = flag.alloc(sizeof(int32_t));
  if (rc) return rc;
  DAXHIP_CHECK(hipMemsetAsync(flag.p, 0, sizeof(int32_t), s));
  const dim3 g((unsigned)ceil_div(n_cells, 256)), b(256);
  if (aligned16(d_cells))
    k_count<NV, true><<<g, b, 0, s>>>(d_cells, n_cells, d_field, n_points, iso, d_counts,
                                      (int32_t*)flag.p);
  else
    k_count<NV, false><<<g, b, 0, s>>>(d_cells, n_cells, d_field, n_points, iso, d_counts,
                                       (int32_t*)flag.p);
  DAXHIP_LAUNCH_CHECK("k_count");
  if ((rc = alg::scan_exclusive_i32_async(d_counts, d_offsets, n_cells, s))) return rc;
  TempBuf res(s);  // {total, bad} read back together
  if ((rc = res.alloc(2 * sizeof(int32_t)))) return rc;
  k_count_result<<<1, 64, 0, s>>>(d_offsets, d_counts, n_cells, (const int32_t*)flag.p,
                                  (int32_t*)res.p);
  DAXHIP_LAUNCH_CHECK("k_count_result");
  int32_t h_res[2] = {0, 0};
  DAXHIP_CHECK(hipMemcpyAsync(h_res, res.p, sizeof(h_res), hipMemcpyDeviceToHost, s));
  DAXHIP_CHECK(hipStreamSynchronize(s));
  const int32_t total = h_res[0], bad = h_res[1];
  if (bad) {
    set_error("%s: a cell references a point outside [0, %lld)", name, (long long)n_points);
    return DAX_HIP_BAD_VALUE;
  }
  *h_tris = total;
  return DAX_HIP_OK;
}

inline size_t scratch_bytes(int64_t n_tris) {
  return n_tris > 0 ? (size_t)n_tris * 3 * 2 * sizeof(uint64_t) : 0;
}

// Dedup by sorting, for edges the rows cannot hold: the pairs in the scratch
// become keys A * P + B sorted in place over the bits that can be set,
// carrying their corner indices; the runs of equal keys are the points.
int sort_corners(void* d_scratch, int64_t n_tris, const float* d_field, const float* d_points,
                 int64_t n_points, float iso, float* d_vertices, int32_t* d_conn,
                 int32_t* d_first, int32_t* d_second, float* d_weight, int64_t* h_points,
                 hipStream_t s) {
  const int64_t n = 3 * n_tris;
  uint64_t* sorted = (uint64_t*)d_scratch;
  int32_t* idx = (int32_t*)(sorted + n);
  const dim3 b(256);
  k_pair_keys<<<dim3((unsigned)ceil_div(n, 256)), b, 0, s>>>(sorted, n, (uint64_t)n_points, idx);
  DAXHIP_LAUNCH_CHECK("k_pair_keys");
  const dim3 gn((unsigned)ceil_div(n, 256));
  // keys < P^2: sort over the bits that can be set
  const uint64_t kmax = (uint64_t)n_points * (uint64_t)n_points - 1;
  const int bits = kmax ? 64 - __builtin_clzll(kmax) : 1;
  int rc = alg::sort_u64_bits(sorted, n, bits, s, idx);
  if (rc) return rc;
  // unique points: the runs of equal sorted keys, numbered by a scan of the
  // run starts (the reference's Unique); each corner's point is its run's
  // number (the reference's LowerBounds)
  TempBuf rk(s);
  if ((rc = rk.alloc((size_t)n * sizeof(int32_t)))) return rc;
  int32_t* rank = (int32_t*)rk.p;
  k_run_starts<<<gn, b, 0, s>>>(sorted, n, rank);
  DAXHIP_LAUNCH_CHECK("k_run_starts");
  int32_t u = 0;
  if ((rc = dax_hip_scan_exclusive_i32(rank, rank, n, &u, (void*)s))) return rc;
  k_points<<<gn, b, 0, s>>>(sorted, rank, n, (uint64_t)n_points, d_field, d_points, iso, d_first,
                            d_second, d_weight, d_vertices);
  DAXHIP_LAUNCH_CHECK("k_points");
  k_corner_points<<<gn, b, 0, s>>>(sorted, idx, rank, n, d_conn);
  DAXHIP_LAUNCH_CHECK("k_corner_points");
  *h_points = u;
  return DAX_HIP_OK;
}

// Temporaries of one dedup: its buffers in one block.  The bytes that note
// lower endpoints, the state and the tiles' counts are cleared before the
// corners are noted.
struct Dedup {
  TempBuf buf;
  uint8_t* used = nullptr;  // null: no room for the tables, sort
  DedupState* state = nullptr;
  uint32_t *count = nullptr, *sizes = nullptr, *ptile = nullptr, *n_list = nullptr,
           *n_edges = nullptr;
  PointWord* pw = nullptr;
  uint2* row_place = nullptr;
  TileCorner* list = nullptr;
  int64_t nw = 0, npt = 0, n_tiles = 0;
  explicit Dedup(hipStream_t s) : buf(s) {}

  // 60 bytes a triangle and a byte and a quarter a point; where there is no such
  // memory the sort is left, which takes 48 a triangle.
  int begin(int64_t n_tris, int64_t n_points, hipStream_t s) {
    const int64_t n = 3 * n_tris;
    nw = ceil_div(n_points, 64);
    npt = ceil_div(nw, (int64_t)kPointTile);
    n_tiles = ceil_div(std::min(n_points, n), (int64_t)kRowTile);
    size_t at = 0;
    auto take = [&](size_t bytes) {
      const size_t o = at;
      at = align_up(at + bytes, 256);
      return o;
    };
    const size_t used_at = take((size_t)nw * 64), state_at = take(sizeof(DedupState));
    const size_t count_at = take((size_t)n_tiles * 4);
    const size_t clear = at;
    const size_t pw_at = take((size_t)nw * sizeof(PointWord)), pt_at = take((size_t)npt * 4);
    const size_t nl_at = take(8), ne_at = take(8), sizes_at = take((size_t)n_tiles * 4);
    const size_t rp_at = take((size_t)n * sizeof(uint2));
    const size_t list_at = take((size_t)n * sizeof(TileCorner));
    const int rc = buf.alloc(at);
    if (rc == DAX_HIP_OOM) return DAX_HIP_OK;
    if (rc) return rc;
    char* p = (char*)buf.p;
    used = (uint8_t*)(p + used_at);
    state = (DedupState*)(p + state_at);
    count = (uint32_t*)(p + count_at);
    pw = (PointWord*)(p + pw_at);
    ptile = (uint32_t*)(p + pt_at);
    n_list = (uint32_t*)(p + nl_at);
    n_edges = (uint32_t*)(p + ne_at);
    sizes = (uint32_t*)(p + sizes_at);
    row_place = (uint2*)(p + rp_at);
    list = (TileCorner*)(p + list_at);
    const int64_t n16 = (int64_t)(clear / 16);
    k_clear16<<<dim3((unsigned)ceil_div(n16, 256)), dim3(256), 0, s>>>((uint4*)p, n16);
    DAXHIP_LAUNCH_CHECK("k_clear16");
    return DAX_HIP_OK;
  }
};

// The scratch holds the corners' pairs and, in its second half, the tiles'
// distinct edges.
int dedup_corners(Dedup& d, void* d_scratch, int64_t n_tris, const float* d_field,
                  const float* d_points, int64_t n_points, float iso, float* d_vertices,
                  int32_t* d_conn, int32_t* d_first, int32_t* d_second, float* d_weight,
                  int64_t* h_points, hipStream_t s) {
  const int64_t n = 3 * n_tris;
  const int2* pairs = (const int2*)d_scratch;
  int2* edges = (int2*)d_scratch + n;
  const dim3 b(256), gn((unsigned)ceil_div(n, 256));
  // grids over the tiles loop: how many there are is known on the device only
  const dim3 gt((unsigned)std::min<int64_t>(d.n_tiles, 4096));
  const dim3 gl((unsigned)ceil_div(n, kListCorners));
  bool sort = !d.used;
  if (!sort) {
    HostSlot slot(s);
    k_point_prefix<<<dim3((unsigned)d.npt), dim3(kPointTile), 0, s>>>(d.used, d.pw, d.nw, d.ptile);
    DAXHIP_LAUNCH_CHECK("k_point_prefix");
    k_scan_block<<<1, kScanBlock, 0, s>>>(d.ptile, d.npt, nullptr, &d.state->rows, nullptr, nullptr);
    DAXHIP_LAUNCH_CHECK("k_scan_block");
    k_corner_rows<<<gl, b, 0, s>>>(pairs, n, n_points, d.pw, d.ptile, d.count, d.row_place,
                                   d.state);
    DAXHIP_LAUNCH_CHECK("k_corner_rows");
    k_scan_block<<<1, kScanBlock, 0, s>>>(d.count, d.n_tiles, &d.state->rows, d.n_list, nullptr,
                                          nullptr);
    DAXHIP_LAUNCH_CHECK("k_scan_block");
    k_list_corners<<<gn, b, 0, s>>>(pairs, n, d.row_place, d.count, d.state, d.list);
    DAXHIP_LAUNCH_CHECK("k_list_corners");
    k_tile_edges<<<gt, b, 0, s>>>(pairs, d.list, d.count, d.n_list, edges, d.sizes, d.state,
                                  d.row_place);
    DAXHIP_LAUNCH_CHECK("k_tile_edges");
    k_scan_block<<<1, kScanBlock, 0, s>>>(d.sizes, d.n_tiles, &d.state->rows, d.n_edges,
                                          &d.state->overflow, slot.p);
    DAXHIP_LAUNCH_CHECK("k_scan_block");
    k_tile_points<<<gt, b, 0, s>>>(edges, d.count, d.n_list, d.state, d.sizes, d.n_edges, n,
                                   d_field, d_points, iso, d_first, d_second, d_weight, d_vertices);
    DAXHIP_LAUNCH_CHECK("k_tile_points");
    k_number_corners<<<gn, b, 0, s>>>(n, d.state, d.sizes, d.row_place, d_conn);
    DAXHIP_LAUNCH_CHECK("k_number_corners");
    uint32_t u = 0, over = 0;
    if (!slot.p) {
      DAXHIP_CHECK(hipMemcpyAsync(&u, d.n_edges, 4, hipMemcpyDeviceToHost, s));
      DAXHIP_CHECK(hipMemcpyAsync(&over, &d.state->overflow, 4, hipMemcpyDeviceToHost, s));
    }
    DAXHIP_CHECK(slot.wait());
    if (slot.p) {
      u = (uint32_t)((volatile int64_t*)slot.p)[0];
      over = (uint32_t)((volatile int64_t*)slot.p)[1];
    }
    *h_points = u;
    sort = over != 0u;
    if (sort) d.buf.release();
  }
  if (!sort) return DAX_HIP_OK;
  return sort_corners(d_scratch, n_tris, d_field, d_points, n_points, iso, d_vertices, d_conn,
                      d_first, d_second, d_weight, h_points, s);
}

template <int NV>
int generate_cells(const char* name, const int32_t* d_cells, int64_t n_cells, const float* d_field,
                   const float* d_points, int64_t n_points, float iso, unsigned flags,
                   const int32_t* d_counts, const int32_t* d_offsets, int64_t n_tris,
                   void* d_scratch, size_t scratch_bytes_, float* d_vertices, int32_t* d_conn,
                   int32_t* d_first, int32_t* d_second, float* d_weight, int64_t* h_points,
                   void* stream) {
  const bool dedup = (flags & DAX_HIP_MC_DEDUP) != 0;
  if (n_cells < 0 || n_tris < 0 || 3 * n_tris > 0x7fffffffLL || !h_points || n_points < 0 ||
      n_points > 0x7fffffffLL || (flags & ~(unsigned)DAX_HIP_MC_DEDUP) ||
      (n_tris > 0 && (!d_cells || !d_field || !d_points || !d_counts || !d_offsets ||
                      !d_vertices || !d_conn)) ||
      (!dedup && n_tris > 0 && (!d_first || !d_second || !d_weight)) ||
      (dedup && n_tris > 0 && (!d_scratch || scratch_bytes_ < scratch_bytes(n_tris)))) {
    set_error("%s: bad arguments (only DAX_HIP_MC_DEDUP; dedup needs %zu bytes of scratch)", name,
              scratch_bytes(n_tris));
    return DAX_HIP_BAD_VALUE;
  }
  *h_points = 0;
  if (n_tris == 0) return DAX_HIP_OK;
  hipStream_t s = (hipStream_t)stream;
  const dim3 gt((unsigned)ceil_div(n_tris, 256)), b(256);
  const bool vec = aligned16(d_cells);
  Dedup dd(s);
  if (dedup)
    if (const int rc = dd.begin(n_tris, n_points, s)) return rc;
  int2* pairs = dedup ? (int2*)d_scratch : nullptr;
#define DAXHIP_UGEN(VEC)                                                                        \
  k_generate<NV, VEC><<<gt, b, 0, s>>>(d_cells, n_cells, d_field, d_points, n_points, iso,      \
                                       n_tris, d_offsets, pairs, dd.used, d_first, d_second,     \
                                       d_weight, d_vertices, d_conn)
  if (vec)
    DAXHIP_UGEN(true);
  else
    DAXHIP_UGEN(false);
#undef DAXHIP_UGEN
  DAXHIP_LAUNCH_CHECK("k_generate");
  if (!dedup) {
    *h_points = 3 * n_tris;
    return DAX_HIP_OK;
  }
  return dedup_corners(dd, d_scratch, n_tris, d_field, d_points, n_points, iso, d_vertices, d_conn,
                       d_first, d_second, d_weight, h_points, s);
}

// ---- count and generate by blocks of cells: host -----------------------------
inline int64_t cell_blocks(int64_t n_cells) { return ceil_div(n_cells, (int64_t)kCellBlock); }
inline size_t blocks_workspace(int64_t n_cells) {
  return n_cells > 0 ? (size_t)cell_blocks(n_cells) * (kCellWords * 8 + 4) : 0;
}

template <int NV>
int count_blocks(const char* name, const int32_t* d_cells, int64_t n_cells, const float* d_field,
                 int64_t n_points, float iso, void* d_ws, size_t ws_bytes, int64_t* h_tris,
                 hipStream_t s) {
  if (n_cells < 0 || n_points < 0 || n_points > 0x7fffffffLL || !h_tris ||
      n_cells > 0x7fffffffLL / NV || ws_bytes < blocks_workspace(n_cells) ||
      (n_cells > 0 && (!d_cells || !d_field || !d_ws))) {
    set_error("%s: bad arguments", name);
    return DAX_HIP_BAD_VALUE;
  }
  *h_tris = 0;
  if (n_cells == 0) return DAX_HIP_OK;
  const int64_t nb = cell_blocks(n_cells);
  uint64_t* bits = (uint64_t*)d_ws;
  uint32_t* sums = (uint32_t*)(bits + nb * kCellWords);
  const dim3 g((unsigned)nb), b(256);
  if (aligned16(d_cells))
    k_count_blocks<NV, true><<<g, b, 0, s>>>(d_cells, n_cells, d_field, n_points, iso, bits, sums);
  else
    k_count_blocks<NV, false><<<g, b, 0, s>>>(d_cells, n_cells, d_field, n_points, iso, bits, sums);
  DAXHIP_LAUNCH_CHECK("k_count_blocks");
  HostSlot slot(s);
  TempBuf res(s);
  if (!slot.p)
    if (const int rc = res.alloc(16)) return rc;
  k_scan_block<<<1, kScanBlock, 0, s>>>(sums, nb, nullptr, (uint32_t*)res.p, nullptr, slot.p);
  DAXHIP_LAUNCH_CHECK("k_scan_block");
  uint32_t h[2] = {0, 0};
  if (!slot.p) DAXHIP_CHECK(hipMemcpyAsync(h, res.p, sizeof(h), hipMemcpyDeviceToHost, s));
  DAXHIP_CHECK(slot.wait());
  const volatile int64_t* v = slot.p;
  if (v ? v[1] != 0 : h[1] != 0) {
    set_error("%s: a cell references a point outside [0, %lld)", name, (long long)n_points);
    return DAX_HIP_BAD_VALUE;
  }
  *h_tris = v ? v[0] : (int64_t)h[0];
  return DAX_HIP_OK;
}

template <int NV>
int generate_blocks(const char* name, const int32_t* d_cells, int64_t n_cells,
                    const float* d_field, const float* d_points, int64_t n_points, float iso,
                    unsigned flags, const void* d_ws, size_t ws_bytes, int64_t n_tris,
                    void* d_scratch, size_t scratch_bytes_, float* d_vertices, int32_t* d_conn,
                    int32_t* d_first, int32_t* d_second, float* d_weight, int64_t* h_points,
                    hipStream_t s) {
  const bool dedup = (flags & DAX_HIP_MC_DEDUP) != 0;
  if (n_cells < 0 || n_tris < 0 || 3 * n_tris > 0x7fffffffLL || !h_points || n_points < 0 ||
      n_points > 0x7fffffffLL || (flags & ~(unsigned)DAX_HIP_MC_DEDUP) ||
      ws_bytes < blocks_workspace(n_cells) ||
      (n_tris > 0 && (!d_cells || !d_field || !d_points || !d_ws || !d_vertices || !d_conn)) ||
      (!dedup && n_tris > 0 && (!d_first || !d_second || !d_weight)) ||
      (dedup && n_tris > 0 && (!d_scratch || scratch_bytes_ < scratch_bytes(n_tris)))) {
    set_error("%s: bad arguments (only DAX_HIP_MC_DEDUP; dedup needs %zu bytes of scratch)", name,
              scratch_bytes(n_tris));
    return DAX_HIP_BAD_VALUE;
  }
  *h_points = 0;
  if (n_tris == 0) return DAX_HIP_OK;
  const int64_t nb = cell_blocks(n_cells);
  const uint64_t* bits = (const uint64_t*)d_ws;
  const uint32_t* sums = (const uint32_t*)(bits + nb * kCellWords);
  Dedup dd(s);
  if (dedup)
    if (const int rc = dd.begin(n_tris, n_points, s)) return rc;
  const dim3 g((unsigned)ceil_div(nb, 4)), b(256);
#define DAXHIP_BGEN(VEC, DEDUP)                                                                  \
  k_generate_blocks<NV, VEC, DEDUP><<<g, b, 0, s>>>(                                             \
      d_cells, nb, d_field, d_points, iso, n_tris, bits, sums, (int2*)d_scratch, dd.used,        \
      d_first, d_second, d_weight, d_vertices, d_conn)
  const bool vec = aligned16(d_cells);
  if (dedup) {
    if (vec) DAXHIP_BGEN(true, true);
    else DAXHIP_BGEN(false, true);
  } else {
    if (vec) DAXHIP_BGEN(true, false);
    else DAXHIP_BGEN(false, false);
  }
#undef DAXHIP_BGEN
  DAXHIP_LAUNCH_CHECK("k_generate_blocks");
  if (!dedup) {
    *h_points = 3 * n_tris;
    return DAX_HIP_OK;
  }
  return dedup_corners(dd, d_scratch, n_tris, d_field, d_points, n_points, iso, d_vertices, d_conn,
                       d_first, d_second, d_weight, h_points, s);
}

}  // namespace ucell
}  // namespace daxhip

using namespace daxhip;
using namespace daxhip::ucell;

extern "C" {

int dax_hip_mt_count(const int32_t* d_tets, int64_t n_tets, const float* d_field,
                     int64_t n_points, float iso, int32_t* d_counts, int32_t* d_offsets,
                     int64_t* h_tris, void* stream) {
  return count_cells<4>("dax_hip_mt_count", d_tets, n_tets, d_field, n_points, iso, d_counts,
                        d_offsets, h_tris, stream);
}

size_t dax_hip_mt_scratch_bytes(int64_t n_tris) { return scratch_bytes(n_tris); }

int dax_hip_mt_generate(const int32_t* d_tets, int64_t n_tets, const float* d_field,
                        const float* d_points, int64_t n_points, float iso, unsigned flags,
                        const int32_t* d_counts, const int32_t* d_offsets, int64_t n_tris,
                        void* d_scratch, size_t scratch_bytes_, float* d_vertices,
                        int32_t* d_conn, int32_t* d_first, int32_t* d_second, float* d_weight,
                        int64_t* h_points, void* stream) {
  return generate_cells<4>("dax_hip_mt_generate", d_tets, n_tets, d_field, d_points, n_points, iso,
                           flags, d_counts, d_offsets, n_tris, d_scratch, scratch_bytes_,
                           d_vertices, d_conn, d_first, d_second, d_weight, h_points, stream);
}

int dax_hip_mc_hex_count(const int32_t* d_hexes, int64_t n_hexes, const float* d_field,
                         int64_t n_points, float iso, int32_t* d_counts, int32_t* d_offsets,
                         int64_t* h_tris, void* stream) {
  return count_cells<8>("dax_hip_mc_hex_count", d_hexes, n_hexes, d_field, n_points, iso,
                        d_counts, d_offsets, h_tris, stream);
}

size_t dax_hip_mc_hex_scratch_bytes(int64_t n_tris) { return scratch_bytes(n_tris); }

int dax_hip_mc_hex_generate(const int32_t* d_hexes, int64_t n_hexes, const float* d_field,
                            const float* d_points, int64_t n_points, float iso, unsigned flags,
                            const int32_t* d_counts, const int32_t* d_offsets, int64_t n_tris,
                            void* d_scratch, size_t scratch_bytes_, float* d_vertices,
                            int32_t* d_conn, int32_t* d_first, int32_t* d_second,
                            float* d_weight, int64_t* h_points, void* stream) {
  return generate_cells<8>("dax_hip_mc_hex_generate", d_hexes, n_hexes, d_field, d_points,
                           n_points, iso, flags, d_counts, d_offsets, n_tris, d_scratch,
                           scratch_bytes_, d_vertices, d_conn, d_first, d_second, d_weight,
                           h_points, stream);
}

size_t dax_hip_cells_workspace_bytes(int64_t n_cells) { return blocks_workspace(n_cells); }

int dax_hip_mt_count_cells(const int32_t* d_tets, int64_t n_tets, const float* d_field,
                           int64_t n_points, float iso, void* d_workspace, size_t workspace_bytes,
                           int64_t* h_tris, void* stream) {
  return count_blocks<4>("dax_hip_mt_count_cells", d_tets, n_tets, d_field, n_points, iso,
                         d_workspace, workspace_bytes, h_tris, (hipStream_t)stream);
}

int dax_hip_mt_generate_cells(const int32_t* d_tets, int64_t n_tets, const float* d_field,
                              const float* d_points, int64_t n_points, float iso, unsigned flags,
                              const void* d_workspace, size_t workspace_bytes, int64_t n_tris,
                              void* d_scratch, size_t scratch_bytes_, float* d_vertices,
                              int32_t* d_conn, int32_t* d_first, int32_t* d_second,
                              float* d_weight, int64_t* h_points, void* stream) {
  return generate_blocks<4>("dax_hip_mt_generate_cells", d_tets, n_tets, d_field, d_points,
                            n_points, iso, flags, d_workspace, workspace_bytes, n_tris, d_scratch,
                            scratch_bytes_, d_vertices, d_conn, d_first, d_second, d_weight,
                            h_points, (hipStream_t)stream);
}

int dax_hip_mc_hex_count_cells(const int32_t* d_hexes, int64_t n_hexes, const float* d_field,
                               int64_t n_points, float iso, void* d_workspace,
                               size_t workspace_bytes, int64_t* h_tris, void* stream) {
  return count_blocks<8>("dax_hip_mc_hex_count_cells", d_hexes, n_hexes, d_field, n_points, iso,
                         d_workspace, workspace_bytes, h_tris, (hipStream_t)stream);
}

int dax_hip_mc_hex_generate_cells(const int32_t* d_hexes, int64_t n_hexes, const float* d_field,
                                  const float* d_points, int64_t n_points, float iso,
                                  unsigned flags, const void* d_workspace, size_t workspace_bytes,
                                  int64_t n_tris, void* d_scratch, size_t scratch_bytes_,
                                  float* d_vertices, int32_t* d_conn, int32_t* d_first,
                                  int32_t* d_second, float* d_weight, int64_t* h_points,
                                  void* stream) {
  return generate_blocks<8>("dax_hip_mc_hex_generate_cells", d_hexes, n_hexes, d_field, d_points,
                            n_points, iso, flags, d_workspace, workspace_bytes, n_tris, d_scratch,
                            scratch_bytes_, d_vertices, d_conn, d_first, d_second, d_weight,
                            h_points, (hipStream_t)stream);
}

}  // extern "C"
