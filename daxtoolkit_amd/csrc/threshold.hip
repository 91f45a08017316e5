// Threshold: the reference's ThresholdCount (dax/worklet/Threshold.h:30-96,
// a cell passes when every point value v has min <= v <= max) dispatched by
// DispatcherMapCell, and ThresholdTopology (:98-110, the output cell's
// vertices are the input cell's) dispatched by DispatcherGenerateTopology
// (dax/cont/DispatcherGenerateTopology.h:146-256), on a uniform grid (voxels
// become hexahedra with the voxel's corner order) or an unstructured grid of
// one cell shape.
//   count    : per cell 1 or 0 (int32, the reference's dax::Id count)
//   prepare  : exclusive scan of the counts (first output cell of each input
//              cell, the reference's inclusive scan + upper bounds); with
//              duplicate removal the point mask (1 where a kept cell uses the
//              point, FillPointMask :211-229) and its exclusive scan, which
//              is each used point's rank among the used points -- the value
//              the reference gets by Sort/Unique/LowerBounds of the used ids
//              (ResolveDuplicatePoints :231-254)
//   generate : every kept cell writes count x V vertex ids (remapped to the
//              ranks with duplicate removal), every used point its
//              coordinates at its rank (StreamCompact of the coordinates)
// Counts may be any non-negative values (DispatcherGenerateTopology repeats
// a cell count times); Threshold's are 0 or 1.
#include <algorithm>

#include "bit_stream.h"
#include "common.h"

namespace daxhip {
namespace topo {

constexpr int kTX = 64, kTY = 4;  // uniform-grid blocks: 64 x-cells by 4 rows
constexpr int kZRun = 16;         // planes one thread marches through

// How prepare laid out the workspace (its first int): per-cell offsets and
// per-point ranks (any counts, any grid), or bit words with exclusive popcount
// prefixes for counts 0/1: on a uniform grid a bit per cell and per point, 64
// to a word along x (kModeBits), on an unstructured one 64 to a word in index
// order (kModeLinear).
constexpr int kModeCells = 0, kModeBits = 1, kModeLinear = 2;

__device__ __forceinline__ bool in_range(float v, float lo, float hi) {
  return v >= lo && v <= hi;
}

// Uniform grid: thread (i, j) marches over kZRun cell planes keeping the
// lower plane's four in-range flags in registers.
__global__ __launch_bounds__(kTX* kTY) void k_count_uniform(const float* __restrict__ f, int nx,
                                                             int ny, int nz, float lo, float hi,
                                                             int32_t* __restrict__ counts) {
  const int cx = nx - 1, cy = ny - 1, cz = nz - 1;
  const int i = blockIdx.x * kTX + threadIdx.x, j = blockIdx.y * kTY + threadIdx.y;
  const int k0 = blockIdx.z * kZRun;
  if (i >= cx || j >= cy || k0 >= cz) return;
  const int64_t sy = nx, sz = (int64_t)nx * ny;
  const float* p = f + i + sy * j + sz * k0;
  bool a00 = in_range(p[0], lo, hi), a10 = in_range(p[1], lo, hi);
  bool a01 = in_range(p[sy], lo, hi), a11 = in_range(p[sy + 1], lo, hi);
  const int k1 = min(k0 + kZRun, cz);
  int32_t* out = counts + i + (int64_t)cx * (j + (int64_t)cy * k0);
  const int64_t cplane = (int64_t)cx * cy;
#pragma unroll 4
  for (int k = k0; k < k1; ++k) {
    p += sz;
    const bool b00 = in_range(p[0], lo, hi), b10 = in_range(p[1], lo, hi);
    const bool b01 = in_range(p[sy], lo, hi), b11 = in_range(p[sy + 1], lo, hi);
    *out = (a00 && a10 && a01 && a11 && b00 && b10 && b01 && b11) ? 1 : 0;
    out += cplane;
    a00 = b00;
    a10 = b10;
    a01 = b01;
    a11 = b11;
  }
}

// The counts of a wave's 256 cells (lane l holds cells 4l .. 4l+3 as bits
// of `kept`) written through the wave's LDS slice so that each store
// instruction covers 64 consecutive cells; n = cells of the 256 in the row.
__device__ __forceinline__ void store_counts256(int32_t* s_w, unsigned kept, int32_t* out, int n) {
  const int lane = threadIdx.x & 63;
  int4 v;
  v.x = (int)(kept & 1u);
  v.y = (int)((kept >> 1) & 1u);
  v.z = (int)((kept >> 2) & 1u);
  v.w = (int)((kept >> 3) & 1u);
  *(int4*)(s_w + 4 * lane) = v;
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int x = lane + 64 * q;
    const int32_t c = s_w[x];
    if (x < n) out[x] = c;
  }
  __builtin_amdgcn_wave_barrier();
}

// The same with rows of 16-byte aligned float4s (nx % 4 == 0): lane l of a
// wave covers cells x0 .. x0+3 (x0 = 4 * (64 * blockIdx.x + l)) from one
// float4 per point row and the next lane's first value (lane 63 loads it).
// The loads (load_row5) and the range bits (row5_bits) are separate so that
// a plane's rows can be loaded while the previous plane is processed.
struct Row5 {
  float4 v;
  float tail;  // lane 63: the next lane's first value
};

__device__ __forceinline__ Row5 load_row5(const float* __restrict__ row, int x0, int nx) {
  Row5 r;
  r.v = make_float4(0.f, 0.f, 0.f, 0.f);
  r.tail = 0.f;
  if (x0 < nx) r.v = *(const float4*)(row + x0);
  if ((threadIdx.x & 63) == 63 && x0 + 4 < nx) r.tail = row[x0 + 4];
  return r;
}

__device__ __forceinline__ unsigned row5_bits(const Row5& r, float lo, float hi) {
  float nxt = __shfl_down(r.v.x, 1, 64);
  if ((threadIdx.x & 63) == 63) nxt = r.tail;
  return (unsigned)in_range(r.v.x, lo, hi) | (unsigned)in_range(r.v.y, lo, hi) << 1 |
         (unsigned)in_range(r.v.z, lo, hi) << 2 | (unsigned)in_range(r.v.w, lo, hi) << 3 |
         (unsigned)in_range(nxt, lo, hi) << 4;
}

__device__ __forceinline__ unsigned range_bits5(const float* __restrict__ row, int x0, int nx,
                                                float lo, float hi) {
  return row5_bits(load_row5(row, x0, nx), lo, hi);
}

__global__ __launch_bounds__(kTX* kTY) void k_count_uniform4(const float* __restrict__ f, int nx,
                                                              int ny, int nz, float lo, float hi,
                                                              int32_t* __restrict__ counts) {
  const int cx = nx - 1, cy = ny - 1, cz = nz - 1;
  const int x0 = 4 * (blockIdx.x * kTX + threadIdx.x), j = blockIdx.y * kTY + threadIdx.y;
  const int k0 = blockIdx.z * kZRun;
  if (j >= cy || k0 >= cz) return;  // whole waves (one row per wave)
  const int64_t sy = nx, sz = (int64_t)nx * ny;
  const float* p = f + sy * j + sz * k0;
  // bit q: point x0+q in range in both rows j and j+1 of the plane
  __shared__ __align__(16) int32_t s_cnt[kTY][256];
  unsigned a = range_bits5(p, x0, nx, lo, hi) & range_bits5(p + sy, x0, nx, lo, hi);
  const int k1 = min(k0 + kZRun, cz);
  const int xw = 256 * (int)blockIdx.x;  // the wave's first cell
  int32_t* out = counts + xw + (int64_t)cx * (j + (int64_t)cy * k0);
  const int64_t cplane = (int64_t)cx * cy;
  // point plane k + 1 is loaded while plane k is processed (k + 1 <= k1 <= nz - 1)
  p += sz;
  Row5 n0 = load_row5(p, x0, nx), n1 = load_row5(p + sy, x0, nx);
  for (int k = k0; k < k1; ++k) {
    const unsigned b = row5_bits(n0, lo, hi) & row5_bits(n1, lo, hi);
    if (k + 1 < k1) {
      p += sz;
      n0 = load_row5(p, x0, nx);
      n1 = load_row5(p + sy, x0, nx);
    }
    const unsigned both = a & b, kept = both & (both >> 1);  // cell q: points q and q+1
    store_counts256(s_cnt[threadIdx.y], kept, out, min(256, cx - xw));
    out += cplane;
    a = b;
  }
}

// Unstructured grid: a thread per cell of nv vertices (nv <= 8); an id
// outside [0, n_points) sets *bad and counts 0.
__global__ __launch_bounds__(256) void k_count_cells(const int32_t* __restrict__ cells, int nv,
                                                     int64_t n_cells,
                                                     const float* __restrict__ f,
                                                     int64_t n_points, float lo, float hi,
                                                     int32_t* __restrict__ counts,
                                                     int32_t* __restrict__ bad) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n_cells) return;
  bool ok = true, keep = true;
  for (int v = 0; v < nv; ++v) {
    const int32_t id = cells[c * nv + v];
    if (id < 0 || id >= n_points) {
      ok = false;
      break;
    }
    keep = keep && in_range(f[id], lo, hi);
  }
  if (!ok) *bad = 1;
  counts[c] = ok && keep ? 1 : 0;
}

// Uniform grid point mask: point (i, j, k) is used when one of its (up to 8)
// cells has a non-zero count.  A wave per 64 points of a row (blockDim.x is
// the wave), 4 rows per block, marching over z with the lower cell plane's
// result in a register; per plane each lane reads its cell column x = i of
// rows j-1 and j and takes column i-1 from the lane below (lane 0 reads it).
__global__ __launch_bounds__(kTX* kTY) void k_mask_uniform(const int32_t* __restrict__ counts,
                                                            int nx, int ny, int nz,
                                                            int32_t* __restrict__ mask) {
  const int cx = nx - 1, cy = ny - 1, cz = nz - 1;
  const int i = blockIdx.x * kTX + threadIdx.x, j = blockIdx.y * kTY + threadIdx.y;
  const int k0 = blockIdx.z * kZRun;
  if (j >= ny || k0 >= nz) return;  // whole waves (one row per wave)
  const bool lane0 = threadIdx.x == 0;
  const int64_t row_lo = (int64_t)cx * (j - 1), row_hi = (int64_t)cx * j;
  const bool has_lo = j - 1 >= 0, has_hi = j < cy;
  // cell columns x of rows j-1 and j of cell plane kc: any non-zero count
  auto column = [&](const int32_t* q, int x) -> int {
    if (x < 0 || x >= cx) return 0;
    int any = 0;
    if (has_lo) any |= q[row_lo + x] != 0;
    if (has_hi) any |= q[row_hi + x] != 0;
    return any;
  };
  auto plane_any = [&](int kc) -> int {
    const bool ok = kc >= 0 && kc < cz;
    const int32_t* q = counts + (int64_t)cx * cy * (ok ? kc : 0);
    const int own = ok ? column(q, i) : 0;
    int left = __shfl_up(own, 1, 64);
    if (lane0) left = ok ? column(q, i - 1) : 0;
    return own | left;
  };
  int below = plane_any(k0 - 1);
  const int k1 = min(k0 + kZRun, nz);
  int32_t* out = mask + i + (int64_t)nx * (j + (int64_t)ny * k0);
  for (int k = k0; k < k1; ++k) {
    const int above = plane_any(k);
    if (i < nx) *out = below | above;
    out += (int64_t)nx * ny;
    below = above;
  }
}

__global__ __launch_bounds__(256) void k_fill_i32(int32_t* __restrict__ p, int64_t n, int32_t v) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Unstructured point mask: the kept cells store 1 at their vertices (every
// store writes the same value); an id outside [0, n_points) sets *bad.
__global__ __launch_bounds__(256) void k_mark_cells(const int32_t* __restrict__ cells, int nv,
                                                    int64_t n_cells, int64_t n_points,
                                                    const int32_t* __restrict__ counts,
                                                    int32_t* __restrict__ mask,
                                                    int32_t* __restrict__ bad) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n_cells || counts[c] <= 0) return;
  for (int v = 0; v < nv; ++v) {
    const int32_t id = cells[c * nv + v];
    if (id >= 0 && id < n_points)
      mask[id] = 1;
    else
      *bad = 1;
  }
}

// Vertex ids of voxel (i, j, k) in the hexahedron's corner order
// (TopologyUniform.h:139-159).
__device__ __forceinline__ void voxel_ids(int64_t c, int nx, int ny, int64_t* ids) {
  const int cx = nx - 1, cy = ny - 1;
  const int64_t i = c % cx, r = c / cx, j = r % cy, k = r / cy;
  const int64_t p = i + (int64_t)nx * (j + (int64_t)ny * k), sy = nx, sz = (int64_t)nx * ny;
  ids[0] = p;
  ids[1] = p + 1;
  ids[2] = p + 1 + sy;
  ids[3] = p + sy;
  ids[4] = p + sz;
  ids[5] = p + 1 + sz;
  ids[6] = p + 1 + sy + sz;
  ids[7] = p + sy + sz;
}

// Every cell with a non-zero count writes its vertex ids count times at its
// first output cell; with `rank` the ids are the used points' ranks.  A
// thread per 4 consecutive cells (one 16-byte load of their counts when
// `vec`: the counts are 16-byte aligned).
__global__ __launch_bounds__(256) void k_emit(const int32_t* __restrict__ mode, int nv,
                                              const int32_t* __restrict__ cells,
                                              int64_t n_cells, int nx, int ny,
                                              const int32_t* __restrict__ counts, bool vec,
                                              const int32_t* __restrict__ offs,
                                              const int32_t* __restrict__ rank,
                                              int32_t* __restrict__ conn) {
  const int64_t c0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (c0 >= n_cells || *mode != kModeCells) return;
  int cnt[4];
  if (vec && c0 + 4 <= n_cells) {
    const int4 v = *(const int4*)(counts + c0);
    cnt[0] = v.x;
    cnt[1] = v.y;
    cnt[2] = v.z;
    cnt[3] = v.w;
  } else {
    for (int q = 0; q < 4; ++q) cnt[q] = c0 + q < n_cells ? counts[c0 + q] : 0;
  }
  for (int q = 0; q < 4; ++q) {
    const int n = cnt[q];
    if (n <= 0) continue;
    const int64_t c = c0 + q;
    int64_t ids[8];
    if (cells) {
      for (int v = 0; v < nv; ++v) ids[v] = cells[c * nv + v];
    } else {
      voxel_ids(c, nx, ny, ids);
    }
    int32_t out[8];
    for (int v = 0; v < nv; ++v) out[v] = rank ? rank[ids[v]] : (int32_t)ids[v];
    int32_t* dst = conn + (int64_t)offs[c] * nv;
    for (int r = 0; r < n; ++r)
      for (int v = 0; v < nv; ++v) dst[(int64_t)r * nv + v] = out[v];
  }
}

// The mask of points p0 .. p0+3 (one 16-byte load when `vec`).
__device__ __forceinline__ void load_mask4(const int32_t* __restrict__ mask, int64_t p0, int64_t n,
                                           bool vec, int* m) {
  if (vec && p0 + 4 <= n) {
    const int4 v = *(const int4*)(mask + p0);
    m[0] = v.x;
    m[1] = v.y;
    m[2] = v.z;
    m[3] = v.w;
  } else {
    for (int q = 0; q < 4; ++q) m[q] = p0 + q < n ? mask[p0 + q] : 0;
  }
}

// Coordinates of the used points at their ranks: from `points`, or on a
// uniform grid origin + spacing * (i, j, k).  A thread per 4 points.
__global__ __launch_bounds__(256) void k_compact_points(const float* __restrict__ points,
                                                        int64_t n_points, int nx, int ny,
                                                        float ox, float oy, float oz, float hx,
                                                        float hy, float hz,
                                                        const int32_t* __restrict__ mask, bool vec,
                                                        const int32_t* __restrict__ rank,
                                                        const int32_t* __restrict__ mode,
                                                        float* __restrict__ out) {
  const int64_t p0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (p0 >= n_points || *mode != kModeCells) return;
  int m[4];
  load_mask4(mask, p0, n_points, vec, m);
  for (int q = 0; q < 4; ++q) {
    if (!m[q]) continue;
    const int64_t p = p0 + q, u = rank[p];
    float x, y, z;
    if (points) {
      x = points[3 * p];
      y = points[3 * p + 1];
      z = points[3 * p + 2];
    } else {
      const int64_t i = p % nx, r = p / nx, j = r % ny, k = r / ny;
      x = ox + hx * (float)i;
      y = oy + hy * (float)j;
      z = oz + hz * (float)k;
    }
    out[3 * u] = x;
    out[3 * u + 1] = y;
    out[3 * u + 2] = z;
  }
}

// CompactPointField with the ranks of the prepare step: the used points'
// values, in point order (a StreamCompact by the point mask).  A thread per
// 4 points.
__global__ __launch_bounds__(256) void k_compact_values(const uint32_t* __restrict__ in, int words,
                                                        int64_t n_points,
                                                        const int32_t* __restrict__ mask, bool vec,
                                                        const int32_t* __restrict__ rank,
                                                        const int32_t* __restrict__ mode,
                                                        uint32_t* __restrict__ out) {
  const int64_t p0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (p0 >= n_points || *mode != kModeCells) return;
  int m[4];
  load_mask4(mask, p0, n_points, vec, m);
  for (int q = 0; q < 4; ++q) {
    if (!m[q]) continue;
    const int64_t p = p0 + q, u = rank[p];
    for (int w = 0; w < words; ++w) out[u * words + w] = in[p * words + w];
  }
}

inline bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

// ---- bit-word layout (uniform grids, counts 0/1) ----
// Cell words: cell row (j, k) has wcx = ceil(cx / 64) words, word index
// (j + cy * k) * wcx + w.  Point words: point row (j, k) has wpx =
// ceil(nx / 64) words, index (j + ny * k) * wpx + w.  Words come in tiles of
// kWordTile: a word's exclusive popcount prefix is its prefix within the
// tile plus the tile's.
constexpr int kWordTile = 256;

struct BitGeom {
  int nx, ny, nz, cx, cy, cz, wcx, wpx;
  int64_t n_cwords, n_pwords;
  mc::FastDiv div_wcx, div_cy, div_cx, div_wpx, div_ny, div_nx;
};

inline BitGeom bit_geom(int nx, int ny, int nz) {
  BitGeom b;
  b.nx = nx;
  b.ny = ny;
  b.nz = nz;
  b.cx = nx - 1;
  b.cy = ny - 1;
  b.cz = nz - 1;
  b.wcx = (b.cx + 63) / 64;
  b.wpx = (nx + 63) / 64;
  b.n_cwords = (int64_t)b.wcx * b.cy * b.cz;
  b.n_pwords = (int64_t)b.wpx * ny * nz;
  b.div_wcx = mc::make_fast_div((uint32_t)b.wcx);
  b.div_cy = mc::make_fast_div((uint32_t)b.cy);
  b.div_cx = mc::make_fast_div((uint32_t)b.cx);
  b.div_wpx = mc::make_fast_div((uint32_t)b.wpx);
  b.div_ny = mc::make_fast_div((uint32_t)ny);
  b.div_nx = mc::make_fast_div((uint32_t)nx);
  return b;
}

__host__ __device__ __forceinline__ FlatRows cell_rows(const BitGeom& g) {
  return FlatRows{g.cx, g.wcx, g.cx * g.cy * g.cz, g.div_wcx};
}
__host__ __device__ __forceinline__ FlatRows point_rows(const BitGeom& g) {
  return FlatRows{g.nx, g.wpx, g.nx * g.ny * g.nz, g.div_wpx};
}

// Header of the workspace: [0] layout mode, [1] flag of counts outside
// {0, 1}, [2..4] the uniform grid's nx, ny, nz, [5] 1 when prepare computed
// the point ranks (duplicate removal), [6] output cells, [7] used points, [8]
// flag of a cell with a point id out of range.
constexpr int kHeaderInts = 9, kHeaderBadId = 8;

// The words of an unstructured grid: one row of cells, one of points.
inline BitGeom bit_linear(int64_t n_cells, int64_t n_points) {
  BitGeom b;
  b.nx = (int)n_points;
  b.cx = (int)n_cells;
  b.ny = b.nz = b.cy = b.cz = 1;
  b.wcx = (int)((n_cells + 63) / 64);
  b.wpx = (int)((n_points + 63) / 64);
  b.n_cwords = b.wcx;
  b.n_pwords = b.wpx;
  b.div_wcx = mc::make_fast_div((uint32_t)b.wcx);
  b.div_cx = mc::make_fast_div((uint32_t)b.cx);
  b.div_wpx = mc::make_fast_div((uint32_t)b.wpx);
  b.div_nx = mc::make_fast_div((uint32_t)b.nx);
  b.div_cy = b.div_ny = mc::make_fast_div(1u);
  return b;
}

// Words, exclusive popcount prefixes within the tiles and the tiles' (sums,
// then exclusive prefixes) of the cells or the points.
struct WordSet {
  uint64_t* bits;
  int32_t* pre;
  int32_t* tile;
};

// Bits of the points whose value is in range: the field read once as a flat
// stream.  Bound by HBM (512^3: 88 us, 6.1 TB/s).
__global__ __launch_bounds__(256) void k_range_bits(FlatRows rows, int64_t nwords,
                                                    const float* __restrict__ f, float lo,
                                                    float hi, uint64_t* __restrict__ pbits) {
  __shared__ FlatLds<128> sh;
  const int64_t w0 = (int64_t)blockIdx.x * 128;
  classify_flat<128, kFlatLoads>(rows, f, pbits, (uint32_t)w0, (uint32_t)min(w0 + 128, nwords), sh,
                                 [&](float v) { return in_range(v, lo, hi); });
}

// Bits of the non-zero counts; *general = 1 if a count is outside {0, 1}.
__global__ __launch_bounds__(256) void k_count_bits(FlatRows rows, int64_t nwords,
                                                    const int32_t* __restrict__ counts,
                                                    uint64_t* __restrict__ cbits,
                                                    int32_t* __restrict__ general) {
  __shared__ FlatLds<128> sh;
  const int64_t w0 = (int64_t)blockIdx.x * 128;
  bool bad = false;
  classify_flat<128, kFlatLoads>(rows, reinterpret_cast<const float*>(counts), cbits, (uint32_t)w0,
                                 (uint32_t)min(w0 + 128, nwords), sh, [&](float v) {
                                   const int32_t c = __builtin_bit_cast(int32_t, v);
                                   bad = bad || c < 0 || c > 1;
                                   return c != 0;
                                 });
  if (bad) *general = 1;
}

// The tile's words (word w of thread threadIdx.x, 0 past the end): LDS copy,
// popcount prefixes and the tile's sum.  s_w holds kWordTile + 1 words.
__device__ __forceinline__ void store_tile(const WordSet& ws, int64_t w, int64_t nwords,
                                           uint64_t word, bool store_bits, uint64_t* s_w,
                                           uint32_t* s_scan) {
  s_w[threadIdx.x] = word;
  uint32_t total;
  const uint32_t pre = block_excl_scan((uint32_t)__popcll(word), total, s_scan);
  if (w < nwords) {
    if (store_bits) ws.bits[w] = word;
    ws.pre[w] = (int32_t)pre;
  }
  if (threadIdx.x == 0) ws.tile[blockIdx.x] = (int32_t)total;
}

// Cell words from the point words: a cell is kept when its eight points are
// in range, so a word is the AND over its four point rows of p & p >> 1.
// Also the counts as int32: with a column of threads marching over z and
// keeping flags in registers, reads and writes mixed, this and the field
// took 277 us at 512^3; the field's stream and this take 88 + 110.
__global__ __launch_bounds__(kWordTile) void k_cell_words(BitGeom g,
                                                          const uint64_t* __restrict__ pbits,
                                                          WordSet ws,
                                                          int32_t* __restrict__ counts) {
  __shared__ uint64_t s_w[kWordTile + 1];
  __shared__ uint32_t s_scan[kWordTile / 64];
  const uint32_t w0 = blockIdx.x * kWordTile, w = w0 + threadIdx.x;
  uint64_t word = 0ull;
  if (w < (uint32_t)g.n_cwords) {
    const uint32_t row = mc::fast_div(w, g.div_wcx);
    const int wx = (int)(w - row * (uint32_t)g.wcx);
    const uint32_t k = mc::fast_div(row, g.div_cy), j = row - k * (uint32_t)g.cy;
    const bool next = wx + 1 < g.wpx;
    word = mc::low_mask(g.cx - 64 * wx);
#pragma unroll
    for (uint32_t q = 0; q < 4u; ++q) {
      const uint64_t* p = pbits + ((int64_t)(j + (q & 1u)) + (int64_t)g.ny * (k + (q >> 1))) * g.wpx + wx;
      const uint64_t a = p[0], a1 = next ? p[1] : 0ull;
      word &= a & mc::shr1(a, a1);
    }
  }
  store_tile(ws, w, g.n_cwords, word, true, s_w, s_scan);
  store_words_i32(cell_rows(g), g.div_cx, s_w, w0,
                  (uint32_t)min((int64_t)w0 + kWordTile, g.n_cwords), counts);
}

// Popcount prefixes of words already there (with a second row of blocks, of
// two sets).  Nothing where the counts turned out to be general.
__global__ __launch_bounds__(kWordTile) void k_word_prefix(WordSet w0, int64_t n0, WordSet w1,
                                                           int64_t n1,
                                                           const int32_t* __restrict__ general) {
  if (*general) return;  // uniform
  const WordSet ws = blockIdx.y == 0 ? w0 : w1;
  const int64_t nwords = blockIdx.y == 0 ? n0 : n1;
  if ((int64_t)blockIdx.x * kWordTile >= nwords) return;  // uniform
  __shared__ uint64_t s_w[kWordTile + 1];
  __shared__ uint32_t s_scan[kWordTile / 64];
  const int64_t w = (int64_t)blockIdx.x * kWordTile + threadIdx.x;
  store_tile(ws, w, nwords, w < nwords ? ws.bits[w] : 0ull, false, s_w, s_scan);
}

// Point words: point (i, j, k) is used when a cell of cell rows j-1, j in
// cell planes k-1, k at x = i-1 or i is kept, i.e. the word is the OR over
// those four cell rows of c | c << 1 | (the previous word's bit 63).  With
// `mask`, also the int32 mask, streamed out: a wave per point row took 311 us
// at 512^3 (537 MB of mask), this takes 105.
__global__ __launch_bounds__(kWordTile) void k_mask_words(BitGeom g,
                                                          const uint64_t* __restrict__ cbits,
                                                          WordSet ws, int32_t* __restrict__ mask) {
  __shared__ uint64_t s_w[kWordTile + 1];
  __shared__ uint32_t s_scan[kWordTile / 64];
  const uint32_t w0 = blockIdx.x * kWordTile, w = w0 + threadIdx.x;
  uint64_t m = 0ull;
  if (w < (uint32_t)g.n_pwords) {
    const uint32_t row = mc::fast_div(w, g.div_wpx);
    const int wx = (int)(w - row * (uint32_t)g.wpx);
    const int k = (int)mc::fast_div(row, g.div_ny), j = (int)row - k * g.ny;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int jc = j - 1 + (q & 1), kc = k - 1 + (q >> 1);
      if (kc < 0 || kc >= g.cz || jc < 0 || jc >= g.cy) continue;
      const uint64_t* r = cbits + ((int64_t)jc + (int64_t)g.cy * kc) * g.wcx;
      const uint64_t c = wx < g.wcx ? r[wx] : 0ull;     // wx <= wcx
      const uint64_t prev = wx > 0 ? r[wx - 1] : 0ull;  // wx - 1 < wcx
      m |= c | (c << 1) | (prev >> 63);
    }
  }
  store_tile(ws, w, g.n_pwords, m, true, s_w, s_scan);
  if (mask)
    store_words_i32(point_rows(g), g.div_nx, s_w, w0,
                    (uint32_t)min((int64_t)w0 + kWordTile, g.n_pwords), mask);
}

__device__ __forceinline__ uint32_t read_lane(uint32_t v, int l) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}
__device__ __forceinline__ uint64_t read_lane64(uint64_t v, int l) {
  return (uint64_t)read_lane((uint32_t)v, l) | ((uint64_t)read_lane((uint32_t)(v >> 32), l) << 32);
}
// Set bits of the wave-uniform m below the lane's.
__device__ __forceinline__ uint32_t bits_below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// The kept cells' corner ids: a wave takes 64 cell words, each lane loading
// one word and what its cells need (the four point rows' words and
// prefixes), then goes through the words that hold a cell with a lane per
// cell.  All corners of a kept cell are used points, so along x a corner's
// rank is its left neighbour's plus one.  A thread per output cell searching
// the words' prefixes took 139 us at 512^3 (4.4 M cells), this takes 44.
__global__ __launch_bounds__(256) void k_emit_words(BitGeom g, WordSet cells, WordSet pts,
                                                    bool dedup, int64_t n_out, bool vec,
                                                    int32_t* __restrict__ conn) {
  const int lane = threadIdx.x & 63;
  const int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const uint64_t c = w < g.n_cwords ? cells.bits[w] : 0ull;
  uint64_t todo = __ballot(c != 0ull);
  if (!todo) return;
  uint32_t first = 0u, pid = 0u;
  uint64_t mw[4] = {0ull, 0ull, 0ull, 0ull};
  uint32_t mo[4] = {0u, 0u, 0u, 0u};
  if (c) {
    const uint32_t row = mc::fast_div((uint32_t)w, g.div_wcx), wx = (uint32_t)w - row * (uint32_t)g.wcx;
    const uint32_t k = mc::fast_div(row, g.div_cy), j = row - k * (uint32_t)g.cy;
    first = (uint32_t)(cells.tile[w / kWordTile] + cells.pre[w]);
    pid = 64u * wx + (uint32_t)g.nx * (j + (uint32_t)g.ny * k);
    if (dedup) {
#pragma unroll
      for (uint32_t q = 0; q < 4u; ++q) {
        const uint32_t pw = (j + (q & 1u) + (uint32_t)g.ny * (k + (q >> 1))) * (uint32_t)g.wpx + wx;
        mw[q] = pts.bits[pw];
        mo[q] = (uint32_t)(pts.tile[pw / kWordTile] + pts.pre[pw]);
      }
    }
  }
  while (todo) {  // wave-uniform
    const int l = __builtin_ctzll(todo);
    todo &= todo - 1ull;
    const uint64_t cw = read_lane64(c, l);
    const int64_t t = (int64_t)read_lane(first, l) + bits_below(cw);
    uint32_t r[4];
    if (dedup) {
#pragma unroll
      for (int q = 0; q < 4; ++q) r[q] = read_lane(mo[q], l) + bits_below(read_lane64(mw[q], l));
    } else {
      const uint32_t p = read_lane(pid, l) + (uint32_t)lane;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        r[q] = p + (uint32_t)g.nx * ((uint32_t)(q & 1) + (uint32_t)g.ny * (uint32_t)(q >> 1));
    }
    if (((cw >> lane) & 1ull) && t < n_out) {
      const int32_t id[8] = {(int32_t)r[0], (int32_t)r[0] + 1, (int32_t)r[1] + 1, (int32_t)r[1],
                             (int32_t)r[2], (int32_t)r[2] + 1, (int32_t)r[3] + 1, (int32_t)r[3]};
      int32_t* dst = conn + 8 * t;
      if (vec) {
        reinterpret_cast<i32x4*>(dst)[0] = i32x4{id[0], id[1], id[2], id[3]};
        reinterpret_cast<i32x4*>(dst)[1] = i32x4{id[4], id[5], id[6], id[7]};
      } else {
#pragma unroll
        for (int v = 0; v < 8; ++v) dst[v] = id[v];
      }
    }
  }
}

// The used points' coordinates (origin + spacing * ijk) or values (`words`
// 4-byte words of `in`) at their ranks: a wave takes kCompactWords point
// words and goes through those that hold a used point four at a time, a lane
// per point, so that four words' loads are in flight.  A thread per used
// point searching the prefixes took 80 us at 512^3 (4.5 M points), this takes
// 30.
constexpr int kCompactWords = 32;
__global__ __launch_bounds__(256) void k_compact_words(BitGeom g, WordSet pts, int64_t n_used,
                                                       float ox, float oy, float oz, float hx,
                                                       float hy, float hz,
                                                       float* __restrict__ coords,
                                                       const uint32_t* __restrict__ in, int words,
                                                       uint32_t* __restrict__ out) {
  const int lane = threadIdx.x & 63;
  const int64_t w = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * kCompactWords + lane;
  const uint64_t m = lane < kCompactWords && w < g.n_pwords ? pts.bits[w] : 0ull;
  uint64_t todo = __ballot(m != 0ull);
  if (!todo) return;
  uint32_t first = 0u, x0 = 0u, j = 0u, k = 0u;
  if (m) {
    const uint32_t row = mc::fast_div((uint32_t)w, g.div_wpx);
    x0 = 64u * ((uint32_t)w - row * (uint32_t)g.wpx);
    k = mc::fast_div(row, g.div_ny);
    j = row - k * (uint32_t)g.ny;
    first = (uint32_t)(pts.tile[w / kWordTile] + pts.pre[w]);
  }
  while (todo) {  // wave-uniform
    int l[4];
    uint64_t mw[4];
    int64_t u[4];
    bool ok[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      l[b] = todo ? __builtin_ctzll(todo) : 0;
      mw[b] = todo ? read_lane64(m, l[b]) : 0ull;
      todo &= todo - (todo ? 1ull : 0ull);
      u[b] = (int64_t)read_lane(first, l[b]) + bits_below(mw[b]);
      ok[b] = ((mw[b] >> lane) & 1ull) && u[b] < n_used;
    }
    if (coords) {
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        if (!ok[b]) continue;
        const float v[3] = {ox + hx * (float)(int)(read_lane(x0, l[b]) + (uint32_t)lane),
                            oy + hy * (float)(int)read_lane(j, l[b]),
                            oz + hz * (float)(int)read_lane(k, l[b])};
        __builtin_memcpy(coords + 3 * u[b], v, 12);
      }
    } else {
      int64_t p[4];
#pragma unroll
      for (int b = 0; b < 4; ++b)
        p[b] = (int64_t)(read_lane(x0, l[b]) + (uint32_t)lane) +
               (int64_t)g.nx * (read_lane(j, l[b]) + (int64_t)g.ny * read_lane(k, l[b]));
      for (int q = 0; q < words; ++q) {
        uint32_t v[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) v[b] = ok[b] ? in[p[b] * words + q] : 0u;
#pragma unroll
        for (int b = 0; b < 4; ++b)
          if (ok[b]) out[u[b] * words + q] = v[b];
      }
    }
  }
}

// ---- unstructured grids, counts 0/1 ----
// The cells' vertex ids: 16-byte loads for 4 and 8 vertices where the cells
// are 16-byte aligned (NV; 0: any number of vertices, single loads).
template <int NV>
__device__ __forceinline__ void load_ids(const int32_t* __restrict__ cells, int nv, int64_t c,
                                         int32_t* ids) {
  if constexpr (NV != 0) {
#pragma unroll
    for (int q = 0; q < NV / 4; ++q) {
      const i32x4 v = reinterpret_cast<const i32x4*>(cells)[c * (NV / 4) + q];
#pragma unroll
      for (int t = 0; t < 4; ++t) ids[4 * q + t] = v[t];
    }
  } else {
#pragma unroll
    for (int v = 0; v < 8; ++v)
      if (v < nv) ids[v] = cells[c * nv + v];
  }
}

// Zeroes the mask and the header's flags.
__global__ __launch_bounds__(256) void k_clear_linear(int32_t* __restrict__ hdr, int ranked,
                                                      int32_t* __restrict__ mask, int64_t n) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i == 0) {
    hdr[0] = kModeLinear;
    hdr[1] = hdr[2] = hdr[3] = hdr[4] = 0;
    hdr[5] = ranked;
    hdr[kHeaderBadId] = 0;
  }
  if (i + 4 <= n && ((uintptr_t)mask & 15u) == 0) {
    *reinterpret_cast<i32x4*>(mask + i) = i32x4{0, 0, 0, 0};
  } else {
    for (int64_t t = i; t < min(i + 4, n); ++t) mask[t] = 0;
  }
}

// A thread per cell, a wave per cell word: from the points' values whether the
// cell is kept (writing the counts and the word), or (f null) from the word;
// kept cells store 1 in the mask at their vertices.  Bound by the ids (129 MB
// for 4.0 M hexahedra: 29 us, 4.4 TB/s), which are read once: counting (a load
// per id), checking the counts' sum, scanning and marking in passes of their
// own took 67 + 90 + 17 + 15 us.
template <int NV>
__global__ __launch_bounds__(256) void k_cell_range(const int32_t* __restrict__ cells, int nv,
                                                    int64_t n_cells, const float* __restrict__ f,
                                                    int64_t n_points, float lo, float hi,
                                                    int32_t* __restrict__ counts,
                                                    uint64_t* __restrict__ cbits,
                                                    int32_t* __restrict__ mask,
                                                    int32_t* __restrict__ hdr) {
  const int n = NV ? NV : nv;
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const bool there = c < n_cells;
  bool keep = false, ok = true;
  int32_t ids[8];
  if (!f && hdr[1]) return;  // general counts: the words are not theirs
  if (f) {
    if (there) {
      load_ids<NV>(cells, nv, c, ids);
#pragma unroll
      for (int v = 0; v < (NV ? NV : 8); ++v)
        if (v < n) ok = ok && ids[v] >= 0 && ids[v] < n_points;
      keep = ok;
      float x[8];
#pragma unroll
      for (int v = 0; v < (NV ? NV : 8); ++v)
        if (v < n) x[v] = f[ok ? ids[v] : 0];
#pragma unroll
      for (int v = 0; v < (NV ? NV : 8); ++v)
        if (v < n) keep = keep && in_range(x[v], lo, hi);
      counts[c] = keep ? 1 : 0;
    }
    const uint64_t word = __ballot(keep);
    if ((threadIdx.x & 63) == 0 && there) cbits[c >> 6] = word;
  } else if (there && ((cbits[c >> 6] >> (c & 63)) & 1ull)) {
    load_ids<NV>(cells, nv, c, ids);
#pragma unroll
    for (int v = 0; v < (NV ? NV : 8); ++v)
      if (v < n) ok = ok && ids[v] >= 0 && ids[v] < n_points;
    keep = ok;
  }
  if (!ok) hdr[kHeaderBadId] = 1;
  if (keep && mask) {
#pragma unroll
    for (int v = 0; v < (NV ? NV : 8); ++v)
      if (v < n) mask[ids[v]] = 1;
  }
}

// Words of the non-zero mask entries.
__global__ __launch_bounds__(256) void k_mask_bits(FlatRows rows, int64_t nwords,
                                                   const int32_t* __restrict__ mask,
                                                   uint64_t* __restrict__ bits,
                                                   const int32_t* __restrict__ general) {
  __shared__ FlatLds<128> sh;
  if (*general) return;  // uniform
  const int64_t w0 = (int64_t)blockIdx.x * 128;
  classify_flat<128, kFlatLoads>(rows, reinterpret_cast<const float*>(mask), bits, (uint32_t)w0,
                                 (uint32_t)min(w0 + 128, nwords), sh,
                                 [](float v) { return __builtin_bit_cast(int32_t, v) != 0; });
}

// The kept cells' vertex ids, a thread per cell (waves whose word is empty
// leave at once); with `dedup` the used points' ranks, from the point words.
// With a scanned rank per point and an offset per cell, four cells a thread,
// it took 44 us for 4.0 M hexahedra, this 14 (and the scans of 4 bytes a cell
// and a point, 35 us, are of a word per 64).
template <int NV>
__global__ __launch_bounds__(256) void k_emit_linear(const int32_t* __restrict__ cells, int nv,
                                                     int64_t n_cells, int64_t n_points,
                                                     WordSet cs, WordSet ps, bool dedup,
                                                     int64_t n_out, bool vec,
                                                     int32_t* __restrict__ conn) {
  const int n = NV ? NV : nv;
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c >= n_cells) return;
  const int64_t w = c >> 6;
  const uint64_t word = cs.bits[w];
  if (!((word >> (c & 63)) & 1ull)) return;
  const int64_t t = (int64_t)cs.tile[w / kWordTile] + cs.pre[w] +
                    __popcll(word & ((1ull << (c & 63)) - 1ull));
  if (t >= n_out) return;
  int32_t ids[8];
  load_ids<NV>(cells, nv, c, ids);
  if (dedup) {
#pragma unroll
    for (int v = 0; v < (NV ? NV : 8); ++v) {
      if (v >= n || ids[v] < 0 || ids[v] >= n_points) continue;
      const int32_t pw = ids[v] >> 6;
      ids[v] = ps.tile[pw / kWordTile] + ps.pre[pw] +
               __popcll(ps.bits[pw] & ((1ull << (ids[v] & 63)) - 1ull));
    }
  }
  int32_t* dst = conn + t * n;
  if (NV && vec) {
#pragma unroll
    for (int q = 0; q < NV / 4; ++q)
      reinterpret_cast<i32x4*>(dst)[q] =
          i32x4{ids[4 * q], ids[4 * q + 1], ids[4 * q + 2], ids[4 * q + 3]};
  } else {
#pragma unroll
    for (int v = 0; v < (NV ? NV : 8); ++v)
      if (v < n) dst[v] = ids[v];
  }
}

// Exclusive scans of the tiles' sums, block 0 the cells', block 1 the
// points'; the totals go to the header and, with `host`, to pinned memory
// with the header's flags.
constexpr int kSumThreads = 1024;
__global__ __launch_bounds__(kSumThreads) void k_scan_word_tiles(int32_t* __restrict__ ctile,
                                                                 int64_t nc,
                                                                 int32_t* __restrict__ ptile,
                                                                 int64_t np,
                                                                 int32_t* __restrict__ hdr,
                                                                 int64_t* __restrict__ host) {
  __shared__ uint32_t s_scan[kSumThreads / 64];
  uint32_t* t = reinterpret_cast<uint32_t*>(blockIdx.x == 0 ? ctile : ptile);
  const int64_t n = blockIdx.x == 0 ? nc : np;
  uint32_t carry = 0u;
  for (int64_t c0 = 0; c0 < n; c0 += kSumThreads * kScanChunk) {
    const int64_t i0 = c0 + (int64_t)threadIdx.x * kScanChunk;
    u32x4 x[kScanChunk / 4];
    load_chunk(t, i0, n, x);
    uint32_t sum = 0u, total;
#pragma unroll
    for (int q = 0; q < kScanChunk; ++q) sum += x[q / 4][q % 4];
    const uint32_t run = carry + block_excl_scan(sum, total, s_scan);
    carry += total;
    store_prefixes(t, i0, n, x, run);
  }
  if (threadIdx.x == 0) {
    hdr[6 + blockIdx.x] = (int32_t)carry;
    if (host) {
      __hip_atomic_store(host + blockIdx.x, (int64_t)carry, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_SYSTEM);
      if (blockIdx.x == 0) {
        __hip_atomic_store(host + 2, (int64_t)hdr[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(host + 3, (int64_t)hdr[kHeaderBadId], __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
  }
}

// Sum of the caller's per-cell counts in 64 bits (out[0]) and a flag for
// negative counts (out[1]).  The int32 scan of the counts wraps past 2^31-1
// without notice (three counts of 2^31-1 wrap to a positive total), so the
// general path checks the exact sum before it scans.  An atomic per block: with
// one per wave of 2048 blocks they took 102 us for 1.7 M counts, now 10.
__global__ __launch_bounds__(256) void k_count_total_i64(const int32_t* __restrict__ counts,
                                                         int64_t n,
                                                         unsigned long long* __restrict__ out) {
  __shared__ unsigned long long s_sum[4];
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  unsigned long long sum = 0ull;
  bool neg = false;
#pragma unroll 4
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const int32_t c = counts[i];
    neg |= c < 0;
    sum += c > 0 ? (unsigned long long)c : 0ull;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
  if ((threadIdx.x & 63) == 0) s_sum[threadIdx.x >> 6] = sum;
  const bool any_neg = __syncthreads_or(neg);
  if (threadIdx.x == 0) {
    sum = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
    if (sum) atomicAdd(&out[0], sum);
    if (any_neg) atomicOr(&out[1], 1ull);
  }
}

__global__ void k_set_header(int32_t* __restrict__ hdr, int mode, int nx, int ny, int nz,
                             int ranked) {
  if (threadIdx.x == 0) {
    hdr[0] = mode;
    hdr[1] = 0;
    hdr[2] = nx;
    hdr[3] = ny;
    hdr[4] = nz;
    hdr[5] = ranked;
  }
}

// Workspace: a 256-byte header (the layout's mode, a flag), region A (per-
// cell offsets, or cell words and their prefixes), region B (per-point
// ranks, or point words and their prefixes).
constexpr size_t kHeader = 256;

struct TopoWs {
  size_t off_a, off_b, bytes;
};

inline TopoWs topo_ws(int64_t n_cells, int64_t n_points) {
  TopoWs w;
  w.off_a = kHeader;
  w.off_b = w.off_a + align_up((size_t)(n_cells > 0 ? n_cells : 1) * 4, 256);
  w.bytes = w.off_b + align_up((size_t)(n_points > 0 ? n_points : 1) * 4, 256);
  return w;
}

// The bit-word layout inside regions A (cells) and B (points: the in-range
// points' words besides), if it fits there.
struct BitWs {
  size_t cbits, cpre, ctile, mbits, mpre, mtile, pbits;
  int64_t nct, nmt;  // word tiles
  bool fits;
};

inline BitWs bit_ws(const TopoWs& w, const BitGeom& g) {
  BitWs b;
  b.nct = ceil_div(g.n_cwords, (int64_t)kWordTile);
  b.nmt = ceil_div(g.n_pwords, (int64_t)kWordTile);
  b.cbits = w.off_a;
  b.cpre = b.cbits + (size_t)g.n_cwords * 8;
  b.ctile = b.cpre + (size_t)g.n_cwords * 4;
  b.mbits = w.off_b;
  b.pbits = b.mbits + (size_t)g.n_pwords * 8;
  b.mpre = b.pbits + (size_t)g.n_pwords * 8;
  b.mtile = b.mpre + (size_t)g.n_pwords * 4;
  b.fits = b.ctile + (size_t)b.nct * 4 <= w.off_b && b.mtile + (size_t)b.nmt * 4 <= w.bytes;
  return b;
}

inline WordSet cell_set(const void* ws, const BitWs& b) {
  char* p = (char*)const_cast<void*>(ws);
  return WordSet{(uint64_t*)(p + b.cbits), (int32_t*)(p + b.cpre), (int32_t*)(p + b.ctile)};
}
inline WordSet point_set(const void* ws, const BitWs& b) {
  char* p = (char*)const_cast<void*>(ws);
  return WordSet{(uint64_t*)(p + b.mbits), (int32_t*)(p + b.mpre), (int32_t*)(p + b.mtile)};
}

// What a prepare found, as the workspace's header holds it: the layout,
// whether the points were ranked, and the sizes.  The fill calls take it from
// the caller; the generate calls read the header back.
struct Plan {
  int64_t mode, ranked, cells, points, nx, ny, nz, reserved;
};
static_assert(sizeof(Plan) == 64, "eight int64 of the C-ABI's plan");

struct Geometry {  // a uniform grid (cells == nullptr) or an unstructured one
  const int32_t* cells;
  int nv;
  int64_t n_cells, n_points;
  int nx, ny, nz;
};

inline bool uniform_ok(int64_t nx, int64_t ny, int64_t nz) {
  return nx >= 2 && ny >= 2 && nz >= 2 && nx <= 65535 * (int64_t)kTX && ny <= 65535 * kTY &&
         nz <= 65535 * (int64_t)kZRun && nx * ny * nz <= 0x7fffffffLL;
}

// ThresholdCount of a uniform grid (checked arguments).
int count_uniform(const float* d_field, int64_t nx, int64_t ny, int64_t nz, float min_value,
                  float max_value, int32_t* d_counts, hipStream_t s) {
  const int cx = (int)nx - 1, cy = (int)ny - 1, cz = (int)nz - 1;
  if ((nx & 3) == 0 && ((uintptr_t)d_field & 15u) == 0) {
    k_count_uniform4<<<dim3((unsigned)ceil_div(nx, 4 * kTX), (unsigned)ceil_div(cy, kTY),
                            (unsigned)ceil_div(cz, kZRun)),
                       dim3(kTX, kTY), 0, s>>>(
        d_field, (int)nx, (int)ny, (int)nz, min_value, max_value, d_counts);
    DAXHIP_LAUNCH_CHECK("k_count_uniform4");
    return DAX_HIP_OK;
  }
  k_count_uniform<<<dim3((unsigned)ceil_div(cx, kTX), (unsigned)ceil_div(cy, kTY),
                         (unsigned)ceil_div(cz, kZRun)),
                    dim3(kTX, kTY), 0, s>>>(d_field, (int)nx, (int)ny, (int)nz,
                                                              min_value, max_value, d_counts);
  DAXHIP_LAUNCH_CHECK("k_count_uniform");
  return DAX_HIP_OK;
}

// ThresholdCount of an unstructured grid (checked arguments, n_cells > 0).
int count_cells(const Geometry& g, const float* d_field, float min_value, float max_value,
                int32_t* d_counts, hipStream_t s) {
  TempBuf flag(s);
  int rc = flag.alloc(sizeof(int32_t));
  if (rc) return rc;
  DAXHIP_CHECK(hipMemsetAsync(flag.p, 0, sizeof(int32_t), s));
  k_count_cells<<<dim3((unsigned)ceil_div(g.n_cells, 256)), dim3(256), 0, s>>>(
      g.cells, g.nv, g.n_cells, d_field, g.n_points, min_value, max_value, d_counts,
      (int32_t*)flag.p);
  DAXHIP_LAUNCH_CHECK("k_count_cells");
  int32_t bad = 0;
  DAXHIP_CHECK(hipMemcpyAsync(&bad, flag.p, sizeof(int32_t), hipMemcpyDeviceToHost, s));
  DAXHIP_CHECK(hipStreamSynchronize(s));
  if (bad) {
    set_error("dax_hip_threshold_count_cells: a cell references a point outside [0, %lld)",
              (long long)g.n_points);
    return DAX_HIP_BAD_VALUE;
  }
  return DAX_HIP_OK;
}

// Cell words of a uniform grid from its in-range points or from its counts,
// the point words and the totals, read back together.  *general: a count
// outside {0, 1} was found, and nothing else holds.
int prepare_bits(const BitGeom& bg, const BitWs& bw, char* ws, const float* d_field, float lo,
                 float hi, int32_t* d_counts, unsigned flags, int32_t* d_mask, int64_t* cells,
                 int64_t* points, bool* general, hipStream_t s) {
  const bool dedup = (flags & DAX_HIP_MC_DEDUP) != 0;
  int32_t* hdr = (int32_t*)ws;
  const WordSet cs = cell_set(ws, bw), ps = point_set(ws, bw);
  const dim3 b(kWordTile), gc((unsigned)bw.nct);
  k_set_header<<<1, 64, 0, s>>>(hdr, kModeBits, bg.nx, bg.ny, bg.nz, dedup ? 1 : 0);
  DAXHIP_LAUNCH_CHECK("k_set_header");
  if (d_field) {
    uint64_t* pbits = (uint64_t*)(ws + bw.pbits);
    k_range_bits<<<dim3((unsigned)ceil_div(bg.n_pwords, 128)), dim3(256), 0, s>>>(
        point_rows(bg), bg.n_pwords, d_field, lo, hi, pbits);
    DAXHIP_LAUNCH_CHECK("k_range_bits");
    k_cell_words<<<gc, b, 0, s>>>(bg, pbits, cs, d_counts);
    DAXHIP_LAUNCH_CHECK("k_cell_words");
  } else {
    k_count_bits<<<dim3((unsigned)ceil_div(bg.n_cwords, 128)), dim3(256), 0, s>>>(
        cell_rows(bg), bg.n_cwords, d_counts, cs.bits, hdr + 1);
    DAXHIP_LAUNCH_CHECK("k_count_bits");
    k_word_prefix<<<gc, b, 0, s>>>(cs, bg.n_cwords, cs, 0, hdr + 1);
    DAXHIP_LAUNCH_CHECK("k_word_prefix");
  }
  if (dedup) {
    k_mask_words<<<dim3((unsigned)bw.nmt), b, 0, s>>>(
        bg, cs.bits, ps, (flags & DAX_HIP_TOPOLOGY_MASK_OPTIONAL) ? nullptr : d_mask);
    DAXHIP_LAUNCH_CHECK("k_mask_words");
  }
  HostSlot slot(s);
  k_scan_word_tiles<<<dedup ? 2 : 1, kSumThreads, 0, s>>>(cs.tile, bw.nct, ps.tile, bw.nmt, hdr,
                                                          slot.p);
  DAXHIP_LAUNCH_CHECK("k_scan_word_tiles");
  int32_t h[kHeaderInts] = {};
  if (!slot.p)
    DAXHIP_CHECK(hipMemcpyAsync(h, hdr, sizeof(h), hipMemcpyDeviceToHost, s));
  DAXHIP_CHECK(slot.wait());
  const volatile int64_t* v = slot.p;
  *cells = v ? v[0] : h[6];
  *points = !dedup ? 0 : (v ? v[1] : h[7]);
  *general = (v ? v[2] : h[1]) != 0;
  return DAX_HIP_OK;
}

// The same for an unstructured grid, whose kept cells mark their points in
// the mask.  *bad: a kept cell (from a field: any cell) has a point id out of
// range, and nothing else holds.
int prepare_linear(const Geometry& g, const BitGeom& bg, const BitWs& bw, char* ws,
                   const float* d_field, float lo, float hi, int32_t* d_counts, bool dedup,
                   int32_t* d_mask, int64_t* cells, int64_t* points, bool* general, bool* bad,
                   hipStream_t s) {
  int32_t* hdr = (int32_t*)ws;
  const WordSet cs = cell_set(ws, bw), ps = point_set(ws, bw);
  const dim3 b(256), grid((unsigned)ceil_div(g.n_cells, 256));
  int32_t* mask = dedup ? d_mask : nullptr;
  k_clear_linear<<<dim3((unsigned)ceil_div(dedup ? g.n_points : 1, (int64_t)1024)), b, 0, s>>>(
      hdr, dedup ? 1 : 0, mask, dedup ? g.n_points : 0);
  DAXHIP_LAUNCH_CHECK("k_clear_linear");
  if (!d_field) {
    k_count_bits<<<dim3((unsigned)ceil_div(bg.n_cwords, 128)), b, 0, s>>>(
        cell_rows(bg), bg.n_cwords, d_counts, cs.bits, hdr + 1);
    DAXHIP_LAUNCH_CHECK("k_count_bits");
  }
  if (d_field || dedup) {
    const bool vec = aligned16(g.cells);
    auto k = vec && g.nv == 8 ? k_cell_range<8> : (vec && g.nv == 4 ? k_cell_range<4> : k_cell_range<0>);
    k<<<grid, b, 0, s>>>(g.cells, g.nv, g.n_cells, d_field, g.n_points, lo, hi, d_counts, cs.bits,
                         mask, hdr);
    DAXHIP_LAUNCH_CHECK("k_cell_range");
  }
  if (dedup) {
    k_mask_bits<<<dim3((unsigned)ceil_div(bg.n_pwords, 128)), b, 0, s>>>(
        point_rows(bg), bg.n_pwords, d_mask, ps.bits, hdr + 1);
    DAXHIP_LAUNCH_CHECK("k_mask_bits");
  }
  k_word_prefix<<<dim3((unsigned)std::max(bw.nct, dedup ? bw.nmt : 0), dedup ? 2 : 1),
                  dim3(kWordTile), 0, s>>>(cs, bg.n_cwords, ps, bg.n_pwords, hdr + 1);
  DAXHIP_LAUNCH_CHECK("k_word_prefix");
  HostSlot slot(s);
  k_scan_word_tiles<<<dedup ? 2 : 1, kSumThreads, 0, s>>>(cs.tile, bw.nct, ps.tile, bw.nmt, hdr,
                                                          slot.p);
  DAXHIP_LAUNCH_CHECK("k_scan_word_tiles");
  int32_t h[kHeaderInts] = {};
  if (!slot.p) DAXHIP_CHECK(hipMemcpyAsync(h, hdr, sizeof(h), hipMemcpyDeviceToHost, s));
  DAXHIP_CHECK(slot.wait());
  const volatile int64_t* v = slot.p;
  *cells = v ? v[0] : h[6];
  *points = !dedup ? 0 : (v ? v[1] : h[7]);
  *general = (v ? v[2] : h[1]) != 0;
  *bad = (v ? v[3] : h[kHeaderBadId]) != 0;
  return DAX_HIP_OK;
}

// Prepare from the caller's counts, or (d_field) from a field's range with
// the counts written.  The bit-word layouts where they hold, else per-cell
// offsets and per-point ranks.
int prepare(const Geometry& g, const float* d_field, float lo, float hi, int32_t* d_counts,
            unsigned flags, void* d_ws, size_t ws_bytes, int32_t* d_mask, Plan* plan,
            hipStream_t s) {
  const bool dedup = (flags & DAX_HIP_MC_DEDUP) != 0;
  const TopoWs w = topo_ws(g.n_cells, g.n_points);
  if (!d_counts || !plan || !d_ws || ws_bytes < w.bytes || (dedup && !d_mask) ||
      (flags & ~(unsigned)(DAX_HIP_MC_DEDUP | DAX_HIP_TOPOLOGY_MASK_OPTIONAL))) {
    set_error("topology prepare: bad arguments (workspace of %zu bytes needed)", w.bytes);
    return DAX_HIP_BAD_VALUE;
  }
  *plan = Plan{kModeCells, dedup ? 1 : 0, 0, 0, g.nx, g.ny, g.nz, 0};
  char* ws = (char*)d_ws;
  int32_t* hdr = (int32_t*)ws;
  const dim3 b(256);
  int rc = DAX_HIP_OK;
  if (!g.cells) {
    const BitGeom bg = bit_geom(g.nx, g.ny, g.nz);
    const BitWs bw = bit_ws(w, bg);
    if (bw.fits) {
      int64_t cells = 0, points = 0;
      bool general = false;
      if ((rc = prepare_bits(bg, bw, ws, d_field, lo, hi, d_counts, flags, d_mask, &cells, &points,
                             &general, s)))
        return rc;
      if (!general) {
        if (cells * 8 > 0x7fffffffLL) {
          set_error("topology prepare: %lld output cells exceed 2^31 ids", (long long)cells);
          return DAX_HIP_BAD_VALUE;
        }
        plan->mode = kModeBits;
        plan->cells = cells;
        plan->points = points;
        return DAX_HIP_OK;
      }
    } else if (d_field) {
      if ((rc = count_uniform(d_field, g.nx, g.ny, g.nz, lo, hi, d_counts, s))) return rc;
    }
  }
  if (g.cells) {
    const BitGeom bg = bit_linear(g.n_cells, g.n_points);
    const BitWs bw = bit_ws(w, bg);
    // (one row: the end of its last word has to stay an int32)
    if (bw.fits && std::max(g.n_cells, g.n_points) <= 0x7fff0000LL) {
      int64_t cells = 0, points = 0;
      bool general = false, bad = false;
      if ((rc = prepare_linear(g, bg, bw, ws, d_field, lo, hi, d_counts, dedup, d_mask, &cells,
                               &points, &general, &bad, s)))
        return rc;
      if (bad && d_field) {
        set_error("dax_hip_threshold_count_cells: a cell references a point outside [0, %lld)",
                  (long long)g.n_points);
        return DAX_HIP_BAD_VALUE;
      }
      if (bad && !general) {
        set_error("topology prepare: a kept cell references a point outside [0, %lld)",
                  (long long)g.n_points);
        return DAX_HIP_BAD_VALUE;
      }
      if (!general) {
        plan->mode = kModeLinear;
        plan->cells = cells;
        plan->points = points;
        return DAX_HIP_OK;
      }
    } else if (d_field) {
      if ((rc = count_cells(g, d_field, lo, hi, d_counts, s))) return rc;
    }
  }
  k_set_header<<<1, 64, 0, s>>>(hdr, kModeCells, g.nx, g.ny, g.nz, dedup ? 1 : 0);
  DAXHIP_LAUNCH_CHECK("k_set_header");
  // any counts: per-cell offsets and per-point ranks.  The exact sum and the
  // sign of every count are checked first: the scan below is int32.
  {
    TempBuf chk(s);
    if ((rc = chk.alloc(2 * sizeof(unsigned long long)))) return rc;
    unsigned long long* d_chk = (unsigned long long*)chk.p;
    k_fill_i32<<<dim3(1), b, 0, s>>>((int32_t*)d_chk, 4, 0);
    DAXHIP_LAUNCH_CHECK("k_fill_i32");
    if (g.n_cells > 0) {
      const int64_t blocks = std::min<int64_t>(ceil_div(g.n_cells, 256), 512);
      k_count_total_i64<<<dim3((unsigned)blocks), b, 0, s>>>(d_counts, g.n_cells, d_chk);
      DAXHIP_LAUNCH_CHECK("k_count_total_i64");
    }
    unsigned long long h_chk[2] = {0ull, 0ull};
    DAXHIP_CHECK(hipMemcpyAsync(h_chk, d_chk, sizeof(h_chk), hipMemcpyDeviceToHost, s));
    DAXHIP_CHECK(hipStreamSynchronize(s));
    if (h_chk[1]) {
      set_error("topology prepare: a cell count is negative");
      return DAX_HIP_BAD_VALUE;
    }
    if (h_chk[0] > 0x7fffffffull / (unsigned long long)std::max(g.nv, 1)) {
      set_error("topology prepare: %llu output cells of %d vertices exceed 2^31 ids", h_chk[0],
                g.nv);
      return DAX_HIP_BAD_VALUE;
    }
  }
  int32_t* offs = (int32_t*)(ws + w.off_a);
  int32_t* rank = (int32_t*)(ws + w.off_b);
  int32_t total = 0;
  if ((rc = dax_hip_scan_exclusive_i32(d_counts, offs, g.n_cells, &total, s))) return rc;
  plan->cells = total;
  if (!dedup) return DAX_HIP_OK;
  const dim3 gp((unsigned)ceil_div(g.n_points, 256));
  if (g.cells) {
    TempBuf flag(s);
    if ((rc = flag.alloc(sizeof(int32_t)))) return rc;
    k_fill_i32<<<dim3(1), b, 0, s>>>((int32_t*)flag.p, 1, 0);
    DAXHIP_LAUNCH_CHECK("k_fill_i32");
    k_fill_i32<<<gp, b, 0, s>>>(d_mask, g.n_points, 0);
    DAXHIP_LAUNCH_CHECK("k_fill_i32");
    k_mark_cells<<<dim3((unsigned)ceil_div(g.n_cells, 256)), b, 0, s>>>(
        g.cells, g.nv, g.n_cells, g.n_points, d_counts, d_mask, (int32_t*)flag.p);
    DAXHIP_LAUNCH_CHECK("k_mark_cells");
    int32_t bad = 0;
    DAXHIP_CHECK(hipMemcpyAsync(&bad, flag.p, sizeof(int32_t), hipMemcpyDeviceToHost, s));
    DAXHIP_CHECK(hipStreamSynchronize(s));
    if (bad) {
      set_error("topology prepare: a kept cell references a point outside [0, %lld)",
                (long long)g.n_points);
      return DAX_HIP_BAD_VALUE;
    }
  } else {
    k_mask_uniform<<<dim3((unsigned)ceil_div(g.nx, kTX), (unsigned)ceil_div(g.ny, kTY),
                          (unsigned)ceil_div(g.nz, kZRun)),
                     dim3(kTX, kTY), 0, s>>>(d_counts, g.nx, g.ny, g.nz, d_mask);
    DAXHIP_LAUNCH_CHECK("k_mask_uniform");
  }
  int32_t used = 0;
  if ((rc = dax_hip_scan_exclusive_i32(d_mask, rank, g.n_points, &used, s))) return rc;
  plan->points = used;
  return DAX_HIP_OK;
}

// The plan a prepare left in the workspace's header (synchronous).
int read_plan(const void* d_ws, Plan* plan, hipStream_t s) {
  int32_t h[kHeaderInts];
  DAXHIP_CHECK(hipMemcpyAsync(h, d_ws, sizeof(h), hipMemcpyDeviceToHost, s));
  DAXHIP_CHECK(hipStreamSynchronize(s));
  *plan = Plan{h[0], h[5], h[6], h[7], h[2], h[3], h[4], 0};
  return DAX_HIP_OK;
}

// Fills the output grid; `given` is the caller's plan, or null to read the
// header's.
int generate(const Geometry& g, const float* d_points, const float* origin, const float* spacing,
             const int32_t* d_counts, unsigned flags, const void* d_ws, size_t ws_bytes,
             const int32_t* d_mask, const Plan* given, int32_t* d_conn, float* d_coords,
             hipStream_t s) {
  const bool dedup = (flags & DAX_HIP_MC_DEDUP) != 0;
  const TopoWs w = topo_ws(g.n_cells, g.n_points);
  if (!d_counts || !d_ws || ws_bytes < w.bytes || !d_conn || (dedup && (!d_mask || !d_coords)) ||
      (flags & ~(unsigned)DAX_HIP_MC_DEDUP)) {
    set_error("topology generate: bad arguments (workspace of %zu bytes needed)", w.bytes);
    return DAX_HIP_BAD_VALUE;
  }
  const char* ws = (const char*)d_ws;
  const int32_t* hdr = (const int32_t*)ws;
  const int32_t* offs = (const int32_t*)(ws + w.off_a);
  const int32_t* rank = (const int32_t*)(ws + w.off_b);
  float o[3] = {0, 0, 0}, h[3] = {1, 1, 1};
  for (int d = 0; d < 3; ++d) {
    if (origin) o[d] = origin[d];
    if (spacing) h[d] = spacing[d];
  }
  const dim3 b(256);
  // the layout prepare chose, whether it ranked the points, the sizes
  Plan plan;
  if (given) {
    plan = *given;
  } else if (const int rc = read_plan(d_ws, &plan, s)) {
    return rc;
  }
  if (dedup && !plan.ranked) {
    set_error("topology generate: duplicate removal after a prepare without it");
    return DAX_HIP_BAD_VALUE;
  }
  if (plan.mode == kModeCells) {
    k_emit<<<dim3((unsigned)ceil_div(g.n_cells, 1024)), b, 0, s>>>(
        hdr, g.nv, g.cells, g.n_cells, g.nx, g.ny, d_counts, aligned16(d_counts), offs,
        dedup ? rank : nullptr, d_conn);
    DAXHIP_LAUNCH_CHECK("k_emit");
    if (dedup) {
      k_compact_points<<<dim3((unsigned)ceil_div(g.n_points, 1024)), b, 0, s>>>(
          d_points, g.n_points, g.nx, g.ny, o[0], o[1], o[2], h[0], h[1], h[2], d_mask,
          aligned16(d_mask), rank, hdr, d_coords);
      DAXHIP_LAUNCH_CHECK("k_compact_points");
    }
  } else if (plan.mode == kModeLinear && g.cells) {
    const BitGeom bg = bit_linear(g.n_cells, g.n_points);
    const BitWs bw = bit_ws(w, bg);
    if (!bw.fits) {
      set_error("topology generate: workspace of another grid");
      return DAX_HIP_BAD_VALUE;
    }
    const WordSet cs = cell_set(ws, bw), ps = point_set(ws, bw);
    if (plan.cells > 0) {
      const bool vec = aligned16(g.cells);
      auto k = vec && g.nv == 8 ? k_emit_linear<8> : (vec && g.nv == 4 ? k_emit_linear<4> : k_emit_linear<0>);
      k<<<dim3((unsigned)ceil_div(g.n_cells, 256)), b, 0, s>>>(g.cells, g.nv, g.n_cells, g.n_points,
                                                              cs, ps, dedup, plan.cells,
                                                              aligned16(d_conn), d_conn);
      DAXHIP_LAUNCH_CHECK("k_emit_linear");
    }
    if (dedup && plan.points > 0) {
      k_compact_words<<<dim3((unsigned)ceil_div(bg.n_pwords, 4 * kCompactWords)), b, 0, s>>>(
          bg, ps, plan.points, 0, 0, 0, 0, 0, 0, nullptr, (const uint32_t*)d_points, 3,
          (uint32_t*)d_coords);
      DAXHIP_LAUNCH_CHECK("k_compact_words");
    }
  } else if (!g.cells) {
    const BitGeom bg = bit_geom(g.nx, g.ny, g.nz);
    const BitWs bw = bit_ws(w, bg);
    if (!bw.fits || plan.nx != g.nx || plan.ny != g.ny || plan.nz != g.nz) {
      set_error("topology generate: workspace of another grid");
      return DAX_HIP_BAD_VALUE;
    }
    const WordSet cs = cell_set(ws, bw), ps = point_set(ws, bw);
    if (plan.cells > 0) {
      k_emit_words<<<dim3((unsigned)ceil_div(bg.n_cwords, 256)), b, 0, s>>>(
          bg, cs, ps, dedup, plan.cells, aligned16(d_conn), d_conn);
      DAXHIP_LAUNCH_CHECK("k_emit_words");
    }
    if (dedup && plan.points > 0) {
      k_compact_words<<<dim3((unsigned)ceil_div(bg.n_pwords, 4 * kCompactWords)), b, 0, s>>>(
          bg, ps, plan.points, o[0], o[1], o[2], h[0], h[1], h[2], d_coords, nullptr, 0, nullptr);
      DAXHIP_LAUNCH_CHECK("k_compact_words");
    }
  }
  return DAX_HIP_OK;
}

// CompactPointField (checked arguments).
int compact_field(const void* d_in, int words, int64_t n_cells, int64_t n_points, const TopoWs& w,
                  const char* ws,
                  const int32_t* d_mask, const Plan& plan, void* d_out, hipStream_t s) {
  if (!plan.ranked) {
    set_error("dax_hip_topology_compact_point_field: the prepare step did not remove duplicates");
    return DAX_HIP_BAD_VALUE;
  }
  if (plan.mode == kModeBits || plan.mode == kModeLinear) {
    const bool linear = plan.mode == kModeLinear;
    const BitGeom bg = linear ? bit_linear(std::max<int64_t>(n_cells, 1), n_points)
                              : bit_geom((int)plan.nx, (int)plan.ny, (int)plan.nz);
    const BitWs bw = bit_ws(w, bg);
    if ((!linear && plan.nx * plan.ny * plan.nz != n_points) || !bw.fits) {
      set_error("dax_hip_topology_compact_point_field: workspace of another grid");
      return DAX_HIP_BAD_VALUE;
    }
    if (plan.points > 0) {
      k_compact_words<<<dim3((unsigned)ceil_div(bg.n_pwords, 4 * kCompactWords)), dim3(256), 0, s>>>(
          bg, point_set(ws, bw), plan.points, 0, 0, 0, 0, 0, 0, nullptr, (const uint32_t*)d_in,
          words, (uint32_t*)d_out);
      DAXHIP_LAUNCH_CHECK("k_compact_words");
    }
    return DAX_HIP_OK;
  }
  if (!d_mask) {
    set_error("dax_hip_topology_compact_point_field: the point mask is needed for this layout");
    return DAX_HIP_BAD_VALUE;
  }
  k_compact_values<<<dim3((unsigned)ceil_div(n_points, 1024)), dim3(256), 0, s>>>(
      (const uint32_t*)d_in, words, n_points, d_mask, aligned16(d_mask),
      (const int32_t*)(ws + w.off_b), (const int32_t*)ws, (uint32_t*)d_out);
  DAXHIP_LAUNCH_CHECK("k_compact_values");
  return DAX_HIP_OK;
}

}  // namespace topo
}  // namespace daxhip

using namespace daxhip;
using namespace daxhip::topo;

extern "C" {

int dax_hip_threshold_count_uniform(const float* d_field, int64_t nx, int64_t ny, int64_t nz,
                                    float min_value, float max_value, int32_t* d_counts,
                                    void* stream) {
  if (!uniform_ok(nx, ny, nz) || !d_field || !d_counts) {
    set_error("dax_hip_threshold_count_uniform: bad arguments (grid %lld x %lld x %lld)",
              (long long)nx, (long long)ny, (long long)nz);
    return DAX_HIP_BAD_VALUE;
  }
  return count_uniform(d_field, nx, ny, nz, min_value, max_value, d_counts, (hipStream_t)stream);
}

int dax_hip_threshold_count_cells(const int32_t* d_cells, int nv, int64_t n_cells,
                                  const float* d_field, int64_t n_points, float min_value,
                                  float max_value, int32_t* d_counts, void* stream) {
  if (nv < 1 || nv > 8 || n_cells < 0 || n_points < 0 || n_points > 0x7fffffffLL ||
      n_cells > 0x7fffffffLL / nv || (n_cells > 0 && (!d_cells || !d_field || !d_counts))) {
    set_error("dax_hip_threshold_count_cells: bad arguments");
    return DAX_HIP_BAD_VALUE;
  }
  if (n_cells == 0) return DAX_HIP_OK;
  return count_cells(Geometry{d_cells, nv, n_cells, n_points, 0, 0, 0}, d_field, min_value,
                     max_value, d_counts, (hipStream_t)stream);
}

// Geometry of a uniform grid the entry points accept.
#define DAXHIP_UNIFORM_GEOMETRY(name)                                                              \
  if (!uniform_ok(nx, ny, nz)) {                                                                   \
    set_error("%s: unsupported grid %lld x %lld x %lld", name, (long long)nx, (long long)ny,       \
              (long long)nz);                                                                      \
    return DAX_HIP_BAD_VALUE;                                                                      \
  }                                                                                                \
  const Geometry g{nullptr, 8, (nx - 1) * (ny - 1) * (nz - 1), nx * ny * nz, (int)nx, (int)ny,     \
                   (int)nz}

int dax_hip_threshold_plan_uniform(const float* d_field, int64_t nx, int64_t ny, int64_t nz,
                                   float min_value, float max_value, unsigned flags,
                                   int32_t* d_counts, void* d_workspace, size_t workspace_bytes,
                                   int32_t* d_point_mask, int64_t* h_plan8, void* stream) {
  DAXHIP_UNIFORM_GEOMETRY("dax_hip_threshold_plan_uniform");
  if (!d_field) {
    set_error("dax_hip_threshold_plan_uniform: field is NULL");
    return DAX_HIP_BAD_VALUE;
  }
  return prepare(g, d_field, min_value, max_value, d_counts, flags, d_workspace, workspace_bytes,
                 d_point_mask, (Plan*)h_plan8, (hipStream_t)stream);
}

int dax_hip_threshold_prepare_uniform(const float* d_field, int64_t nx, int64_t ny, int64_t nz,
                                      float min_value, float max_value, unsigned flags,
                                      int32_t* d_counts, void* d_workspace,
                                      size_t workspace_bytes, int32_t* d_point_mask,
                                      int64_t* h_cells, int64_t* h_points, void* stream) {
  Plan plan;
  if (!h_cells || !h_points) {
    set_error("dax_hip_threshold_prepare_uniform: h_cells and h_points are required");
    return DAX_HIP_BAD_VALUE;
  }
  *h_cells = *h_points = 0;
  const int rc = dax_hip_threshold_plan_uniform(d_field, nx, ny, nz, min_value, max_value, flags,
                                                d_counts, d_workspace, workspace_bytes,
                                                d_point_mask, (int64_t*)&plan, stream);
  if (rc) return rc;
  *h_cells = plan.cells;
  *h_points = plan.points;
  return DAX_HIP_OK;
}

size_t dax_hip_topology_workspace_bytes(int64_t n_cells, int64_t n_points) {
  return topo_ws(n_cells, n_points).bytes;
}

int dax_hip_topology_plan_uniform(int64_t nx, int64_t ny, int64_t nz, const int32_t* d_counts,
                                  unsigned flags, void* d_workspace, size_t workspace_bytes,
                                  int32_t* d_point_mask, int64_t* h_plan8, void* stream) {
  DAXHIP_UNIFORM_GEOMETRY("dax_hip_topology_prepare_uniform");
  return prepare(g, nullptr, 0.0f, 0.0f, const_cast<int32_t*>(d_counts), flags, d_workspace,
                 workspace_bytes, d_point_mask, (Plan*)h_plan8, (hipStream_t)stream);
}

int dax_hip_topology_prepare_uniform(int64_t nx, int64_t ny, int64_t nz, const int32_t* d_counts,
                                     unsigned flags, void* d_workspace, size_t workspace_bytes,
                                     int32_t* d_point_mask, int64_t* h_cells, int64_t* h_points,
                                     void* stream) {
  Plan plan;
  if (!h_cells || !h_points) {
    set_error("dax_hip_topology_prepare_uniform: h_cells and h_points are required");
    return DAX_HIP_BAD_VALUE;
  }
  *h_cells = *h_points = 0;
  const int rc = dax_hip_topology_plan_uniform(nx, ny, nz, d_counts, flags, d_workspace,
                                               workspace_bytes, d_point_mask, (int64_t*)&plan,
                                               stream);
  if (rc) return rc;
  *h_cells = plan.cells;
  *h_points = plan.points;
  return DAX_HIP_OK;
}

int dax_hip_topology_fill_uniform(int64_t nx, int64_t ny, int64_t nz, const float* h_origin3,
                                  const float* h_spacing3, const int32_t* d_counts,
                                  unsigned flags, const void* d_workspace, size_t workspace_bytes,
                                  const int32_t* d_point_mask, const int64_t* h_plan8,
                                  int32_t* d_conn, float* d_coords, void* stream) {
  DAXHIP_UNIFORM_GEOMETRY("dax_hip_topology_generate_uniform");
  return generate(g, nullptr, h_origin3, h_spacing3, d_counts, flags, d_workspace, workspace_bytes,
                  d_point_mask, (const Plan*)h_plan8, d_conn, d_coords, (hipStream_t)stream);
}

int dax_hip_topology_generate_uniform(int64_t nx, int64_t ny, int64_t nz, const float* h_origin3,
                                      const float* h_spacing3, const int32_t* d_counts,
                                      unsigned flags, const void* d_workspace,
                                      size_t workspace_bytes, const int32_t* d_point_mask,
                                      int32_t* d_conn, float* d_coords, void* stream) {
  return dax_hip_topology_fill_uniform(nx, ny, nz, h_origin3, h_spacing3, d_counts, flags,
                                       d_workspace, workspace_bytes, d_point_mask, nullptr, d_conn,
                                       d_coords, stream);
}

int dax_hip_threshold_plan_cells(const int32_t* d_cells, int nv, int64_t n_cells,
                                 const float* d_field, int64_t n_points, float min_value,
                                 float max_value, unsigned flags, int32_t* d_counts,
                                 void* d_workspace, size_t workspace_bytes, int32_t* d_point_mask,
                                 int64_t* h_plan8, void* stream) {
  if (nv < 1 || nv > 8 || n_cells < 1 || n_points < 1 || n_points > 0x7fffffffLL ||
      n_cells > 0x7fffffffLL / nv || !d_cells || !d_field) {
    set_error("dax_hip_threshold_plan_cells: bad arguments");
    return DAX_HIP_BAD_VALUE;
  }
  const Geometry g{d_cells, nv, n_cells, n_points, 0, 0, 0};
  return prepare(g, d_field, min_value, max_value, d_counts, flags, d_workspace, workspace_bytes,
                 d_point_mask, (Plan*)h_plan8, (hipStream_t)stream);
}

int dax_hip_topology_plan_cells(const int32_t* d_cells, int nv, int64_t n_cells, int64_t n_points,
                                const int32_t* d_counts, unsigned flags, void* d_workspace,
                                size_t workspace_bytes, int32_t* d_point_mask, int64_t* h_plan8,
                                void* stream) {
  if (nv < 1 || nv > 8 || n_cells < 1 || n_points < 1 || n_points > 0x7fffffffLL ||
      n_cells > 0x7fffffffLL / nv || !d_cells) {
    set_error("dax_hip_topology_prepare_cells: bad arguments");
    return DAX_HIP_BAD_VALUE;
  }
  const Geometry g{d_cells, nv, n_cells, n_points, 0, 0, 0};
  return prepare(g, nullptr, 0.0f, 0.0f, const_cast<int32_t*>(d_counts), flags, d_workspace,
                 workspace_bytes, d_point_mask, (Plan*)h_plan8, (hipStream_t)stream);
}

int dax_hip_topology_prepare_cells(const int32_t* d_cells, int nv, int64_t n_cells,
                                   int64_t n_points, const int32_t* d_counts, unsigned flags,
                                   void* d_workspace, size_t workspace_bytes,
                                   int32_t* d_point_mask, int64_t* h_cells, int64_t* h_points,
                                   void* stream) {
  Plan plan;
  if (!h_cells || !h_points) {
    set_error("dax_hip_topology_prepare_cells: h_cells and h_points are required");
    return DAX_HIP_BAD_VALUE;
  }
  *h_cells = *h_points = 0;
  const int rc = dax_hip_topology_plan_cells(d_cells, nv, n_cells, n_points, d_counts, flags,
                                             d_workspace, workspace_bytes, d_point_mask,
                                             (int64_t*)&plan, stream);
  if (rc) return rc;
  *h_cells = plan.cells;
  *h_points = plan.points;
  return DAX_HIP_OK;
}

int dax_hip_topology_fill_cells(const int32_t* d_cells, int nv, int64_t n_cells,
                                const float* d_points, int64_t n_points, const int32_t* d_counts,
                                unsigned flags, const void* d_workspace, size_t workspace_bytes,
                                const int32_t* d_point_mask, const int64_t* h_plan8,
                                int32_t* d_conn, float* d_coords, void* stream) {
  if (nv < 1 || nv > 8 || n_cells < 1 || n_points < 1 || n_points > 0x7fffffffLL ||
      n_cells > 0x7fffffffLL / nv || !d_cells ||
      ((flags & DAX_HIP_MC_DEDUP) && !d_points)) {
    set_error("dax_hip_topology_generate_cells: bad arguments");
    return DAX_HIP_BAD_VALUE;
  }
  const Geometry g{d_cells, nv, n_cells, n_points, 0, 0, 0};
  return generate(g, d_points, nullptr, nullptr, d_counts, flags, d_workspace, workspace_bytes,
                  d_point_mask, (const Plan*)h_plan8, d_conn, d_coords, (hipStream_t)stream);
}

int dax_hip_topology_generate_cells(const int32_t* d_cells, int nv, int64_t n_cells,
                                    const float* d_points, int64_t n_points,
                                    const int32_t* d_counts, unsigned flags,
                                    const void* d_workspace, size_t workspace_bytes,
                                    const int32_t* d_point_mask, int32_t* d_conn,
                                    float* d_coords, void* stream) {
  return dax_hip_topology_fill_cells(d_cells, nv, n_cells, d_points, n_points, d_counts, flags,
                                     d_workspace, workspace_bytes, d_point_mask, nullptr, d_conn,
                                     d_coords, stream);
}

int dax_hip_topology_fill_point_field(const void* d_in, size_t value_bytes, int64_t n_cells,
                                      int64_t n_points, const int32_t* d_point_mask,
                                      const void* d_workspace, size_t workspace_bytes,
                                      const int64_t* h_plan8, void* d_out, void* stream) {
  const TopoWs w = topo_ws(n_cells, n_points);
  if (value_bytes == 0 || value_bytes % 4 || value_bytes > 1024 || n_points < 0 ||
      n_points > 0x7fffffffLL || !d_workspace || workspace_bytes < w.bytes ||
      (n_points > 0 && (!d_in || !d_out))) {
    set_error("dax_hip_topology_compact_point_field: bad arguments (values of 4k bytes, "
              "workspace of %zu bytes)", w.bytes);
    return DAX_HIP_BAD_VALUE;
  }
  if (n_points == 0) return DAX_HIP_OK;
  hipStream_t s = (hipStream_t)stream;
  Plan plan;
  if (h_plan8) {
    plan = *(const Plan*)h_plan8;
  } else if (const int rc = read_plan(d_workspace, &plan, s)) {
    return rc;
  }
  return compact_field(d_in, (int)(value_bytes / 4), n_cells, n_points, w, (const char*)d_workspace,
                       d_point_mask, plan, d_out, s);
}

int dax_hip_topology_compact_point_field(const void* d_in, size_t value_bytes, int64_t n_cells,
                                         int64_t n_points, const int32_t* d_point_mask,
                                         const void* d_workspace, size_t workspace_bytes,
                                         void* d_out, void* stream) {
  return dax_hip_topology_fill_point_field(d_in, value_bytes, n_cells, n_points, d_point_mask,
                                           d_workspace, workspace_bytes, nullptr, d_out, stream);
}

}  // extern "C"
