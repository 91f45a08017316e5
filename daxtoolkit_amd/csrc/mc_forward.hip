// Marching-cubes forward on gfx950: classify -> count/scan -> generate.
//
// Reference path (Kitware/DaxToolkit):
//   MarchingCubesCount          dax/worklet/MarchingCubes.h:53-86
//   ScanInclusive + UpperBounds + visit index
//                               dax/cont/DispatcherGenerateInterpolatedCells.h:180-223
//   MarchingCubesGenerate       dax/worklet/MarchingCubes.h:90-169
//   Sort/Unique/LowerBounds dedup + coordinate interpolation
//                               dax/cont/DispatcherGenerateInterpolatedCells.h:261-301
//
// Design: the field is read once, as one coalesced stream, into inside-bits
// (classify).  Everything topological after that works on the bits: 64 cells
// per 64-bit word op.  Vertex numbering uses active-edge flags in
// (point id, axis) order, which is the order the reference's sort/unique
// produces, so no sort is needed.  The count kernel writes prefixes within
// its blocks and one block scans the blocks' sums; the generate kernel
// revisits only tiles that have output and touches the field only around the
// surface.
//
// Tile shapes (classify unroll and load width, scan sub-tiles, generate tile
// words) are chosen per grid shape by the autotuner at the end of this file.
#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <vector>

#include "mc_kernels.h"

namespace daxhip {
namespace mc {

// Classify the volume's row words.
template <int UNROLL>
__global__ __launch_bounds__(256) void k_classify(VolGeom g, const float* __restrict__ field,
                                                  uint64_t* __restrict__ bits,
                                                  int64_t nwords) {
  const int64_t gtid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  classify_words<UNROLL>(g, field + g.field_off, bits + g.word_off, (gtid >> 6) * UNROLL, nwords);
}

// Rows that are not whole 64-point words, or a field that is not 16-byte
// aligned: TW words per block.  Bound by HBM.
template <int TW>
__global__ __launch_bounds__(256) void k_classify_flat(VolGeom g, const float* __restrict__ field,
                                                       uint64_t* __restrict__ bits,
                                                       int64_t nwords) {
  __shared__ FlatLds<TW> sh;
  const int64_t w0 = (int64_t)blockIdx.x * TW;
  classify_flat<TW, kFlatLoads>(flat_rows(g), field + g.field_off, bits + g.word_off,
                                (uint32_t)w0, (uint32_t)min(w0 + TW, nwords), sh,
                                [&](float v) { return v > g.iso; });
}

template <int UNROLL>
__global__ __launch_bounds__(256) void k_classify_v4(VolGeom g, const float* __restrict__ field,
                                                     uint64_t* __restrict__ bits,
                                                     int64_t nwords) {
  const int64_t gtid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  classify_chunks_v4<UNROLL>(g, field + g.field_off, bits + g.word_off, (gtid >> 6) * UNROLL,
                             nwords);
}

// ---- count and scan --------------------------------------------------------
// 1. k_count: a block of WAVES waves, each wave two count tiles of
//    kCountTile row words (four consecutive words per lane, coalesced loads
//    of the words and their +x/+y/+z neighbours): every word's prefix within
//    its tile, every tile's prefix within the block and output size, and the
//    block's sums.
//    No inter-block dependency.
// 2. k_scan_tsums: one block scans the blocks' sums into exclusive prefixes
//    (the totals after the last) and the 64-bit totals of the control block.
// A word's bases are block + tile + local prefix, formed where they are used
// (stored for every word they were 8 bytes a word more to write, and a launch
// of their own where nothing is generated).
// Dispatch classes of the generate tiles (a byte per tile): 0 heavy (at least
// 5/4 outputs, vertices + triangles, per word), 1 other with output, 2 none.
// tw = 0: no classes (the count blocks do not cover whole generate tiles).
struct TileClasses {
  uint8_t* gcls;
  int tw;
};

template <int WAVES>
__global__ __launch_bounds__(64 * WAVES) void k_count(VolGeom g, const uint64_t* __restrict__ bits,
                                                      uint32_t* __restrict__ lpre,
                                                      unsigned long long* __restrict__ tloc,
                                                      unsigned long long* __restrict__ bsum,
                                                      TileClasses tc, int64_t n_ctiles) {
  constexpr int kBlockTiles = 2 * WAVES;  // count tiles per block
  __shared__ unsigned long long s_ts[kBlockTiles];
  const int wv = threadIdx.x >> 6;
  // XCD-contiguous block order: the block one plane ahead, whose words this
  // block reads as +z neighbours, runs on the same XCD (same L2)
  const int64_t blk = xcd_tile(blockIdx.x, gridDim.x);
  const int64_t pair = blk * WAVES + wv;
  unsigned long long s0 = 0ull, s1 = 0ull;
  if (2 * pair < n_ctiles) count_tile_pair(g, bits + g.word_off, lpre, pair, n_ctiles, s0, s1);
  if ((threadIdx.x & 63) == 0) {
    s_ts[2 * wv] = s0;
    s_ts[2 * wv + 1] = s1;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long run = 0ull;
    for (int i = 0; i < kBlockTiles; ++i) {
      const int64_t tile = blk * kBlockTiles + i;
      if (tile <= n_ctiles) tloc[tile] = run;  // the entry after the last: the totals
      run = add_vt(run, s_ts[i]);
    }
    bsum[blk] = run;
  } else if (threadIdx.x < 64) {  // the block's generate tiles
    const int lane = threadIdx.x;
    auto weight = [&](int first, int n) -> uint32_t {  // outputs of count tiles [first, +n)
      uint32_t w = 0u;
      for (int i = 0; i < n; ++i)
        if (blk * kBlockTiles + first + i < n_ctiles)
          w += (uint32_t)s_ts[first + i] + (uint32_t)(s_ts[first + i] >> 32);
      return w;
    };
    const int l = lane - 1;
    const int cpt = tc.tw / kCountTile;
    if (tc.tw > 0 && l >= 0 && l < kBlockTiles / cpt) {
      const int64_t c0 = blk * kBlockTiles + l * cpt;
      if (c0 < n_ctiles) {
        const uint32_t w = weight(l * cpt, cpt);
        tc.gcls[c0 / cpt] = w == 0u ? 2 : (4ull * w >= 5ull * (uint32_t)tc.tw ? 0 : 1);
      }
    }
  }
}

// Dispatch order of the generate tiles, written by the scan block from the
// count kernel's tile classes: heavy tiles first, then the other tiles with
// output, then the empty ones; within a class, index order.  A grid
// dispatches its blocks roughly in index order as slots free up, so the
// longest tiles start first and the short ones fill the tail (a coarse
// longest-processing-time-first schedule).  Every tile writes at fixed
// offsets, so an order changes no output.  Each thread of the scan block
// takes a contiguous chunk of tiles; two block scans of its class counts
// give its slots.
struct GenOrder {
  const uint8_t* __restrict__ gcls;  // classes of the generate tiles
  int64_t nwords;
  int tw;            // generate tile words: 64, 128, 256, 512 or 1024
  bool gen_classes;  // gcls holds the classes
  uint32_t unit_sp;  // > 0: order units of kOrderUnitTiles tiles a plane (unit_sp tiles) apart
  uint32_t* order;   // [0]: tw (0: no order), [1 + i]: the i-th tile to dispatch
};

// Where the scan reports {T, U} besides the control block (each may be null):
// device memory, and pinned host memory.
struct ScanOut {
  int64_t* counts;
  int64_t* host;
};

constexpr uint32_t kOrderStage = 16384;  // 64 KiB of LDS

// One block scans the count blocks' sums (scan_block_sums), completes the tile
// prefixes and writes the dispatch order.
// LARGE: some thread's chunk exceeds kOrderRegTiles tiles (a separate
// instance, so the common one stays small).
template <bool LARGE>
__global__ __launch_bounds__(kTsumThreads) void k_scan_tsums(const unsigned long long* __restrict__ bsum,
                                                             unsigned long long* __restrict__ bpre,
                                                             int64_t n,
                                                             unsigned long long* __restrict__ tloc,
                                                             int64_t n_ctiles,
                                                             Ctrl* __restrict__ ctrl,
                                                             GenOrder go, int tpb_shift,
                                                             ScanOut so) {
  constexpr int kWaves = kTsumThreads / 64;
  // the scan's wave sums, then the dispatch order's LDS window
  __shared__ uint32_t s_stage[kOrderStage];
  uint32_t* s_v = s_stage;
  uint32_t* s_t = s_stage + kWaves;
  const int tid = threadIdx.x;
  const uint32_t ng = (uint32_t)ceil_div(go.nwords, (int64_t)go.tw);
  const uint32_t Kg = order_chunk(ng, kTsumThreads);
  const bool ordered = go.gen_classes;  // uniform
  const bool units = ordered && go.unit_sp > 0u;
  const uint32_t nunits = units ? ng / kOrderUnitTiles : 0u;
  const uint32_t Ku = units ? order_chunk(nunits, kTsumThreads) : 0u;
  const uint64_t gcls =
      units ? load_unit_classes(go.gcls, Ku, nunits, go.unit_sp)
            : (ordered ? load_classes(go.gcls, (uint32_t)tid * Kg, Kg, ng) : 0ull);

  unsigned long long cv, ct;
  scan_block_sums(bsum, bpre, n, s_v, s_t, cv, ct);
  if (tid == 0) {
    // the count blocks wrote it unless the last one is full
    if ((n_ctiles & ((1 << tpb_shift) - 1)) == 0) tloc[n_ctiles] = 0ull;
    ctrl->total_v = cv;
    ctrl->total_t = ct;
    ctrl->tpb_shift = (uint32_t)tpb_shift;
    if (so.counts) {
      so.counts[0] = (int64_t)ct;
      so.counts[1] = (int64_t)cv;
    }
    if (so.host) {
      __hip_atomic_store(so.host, (int64_t)ct, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      __hip_atomic_store(so.host + 1, (int64_t)cv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }

  if (units)
    write_order_units(gcls, Ku, nunits, go.unit_sp, go.order, (uint32_t)go.tw, s_v, s_t, s_stage,
                      kOrderStage);
  else if (ordered)
    write_order<LARGE>(gcls, go.gcls, Kg, ng, go.order, (uint32_t)go.tw, s_v, s_t, s_stage,
                       kOrderStage);
  else if (tid == 0)
    go.order[0] = 0u;
}

template <int TW, int NT, class Src, bool dedup>
__global__ __launch_bounds__(NT, 4) void k_generate(
    VolGeom g, Src field, const uint64_t* __restrict__ bits, CountSrc cs,
    const Ctrl* __restrict__ ctrl, OutPtrs out, unsigned flags, int64_t cap_points,
    int64_t cap_tris, int64_t* __restrict__ counts, int xcd_order, int64_t tile_lo,
    int64_t ntiles, const uint32_t* __restrict__ order) {
  extern __shared__ uint64_t s_dyn[];
  const bool normals = (flags & DAX_HIP_MC_NORMALS) != 0 && out.normals != nullptr;
  const uint64_t total_v = ctrl->total_v, total_t = ctrl->total_t;
  cs.tpb_shift = (int)ctrl->tpb_shift;
  const uint64_t n_points = dedup ? total_v : 3ull * total_t;
  if (blockIdx.x == 0 && threadIdx.x == 0 && counts) {
    counts[0] = (int64_t)total_t;
    counts[1] = (int64_t)n_points;
  }
  // too many ids for dax::Id or too little room: no output
  if (total_v > 0x7fffffffull || 3ull * total_t > 0x7fffffffull ||
      (int64_t)total_t > cap_tris || (int64_t)n_points > cap_points)
    return;
  // the scan's dispatch order when it was built for this tile size (whole
  // volume launches only), else index order
  uint32_t tag = 0u, ord = 0u;
  if (TW >= kCountTile && order != nullptr) {
    tag = order[0];
    ord = order[1 + blockIdx.x];
  }
  const bool ordered = tag == (uint32_t)TW && (int64_t)(ord & ~kOrderHasOutput) < ntiles;
  const int64_t tile =
      ordered ? (int64_t)(ord & ~kOrderHasOutput)
              : tile_lo + (xcd_order ? xcd_tile(blockIdx.x, ntiles) : (int64_t)blockIdx.x);
  generate_tile<TW, NT, Src, dedup>(g, field, bits + g.word_off, tile * TW, out, normals, 0, 0,
                                    s_dyn, cs, ordered && (ord & kOrderHasOutput) != 0u);
}

// Slice classify: a thread per row word.  Along a row the plane value
// pn0 * ((o0 + s0 * x) - po0) + t1 + t2 (t1, t2: the row's y and z terms)
// is a monotonic function of x: int -> float conversion, multiplication by
// a constant, addition of a constant and their round-to-nearest are all
// monotonic.  So "value > iso" changes at most once along the row, and a
// word whose end points agree is all ones or all zeros; in the others six
// halving steps, each evaluating one point with exactly the operations
// FieldPlane uses, find the change.  Bound by the words' stores (512^3: 16.8
// MB); a wave per 8 rows with a 64-way search per row took 37 us there, this
// takes 11.
__global__ __launch_bounds__(256) void k_classify_plane(VolGeom g, FieldPlane pl,
                                                        uint64_t* __restrict__ bits) {
  const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= g.nwords) return;
  const uint32_t row = fast_div((uint32_t)w, g.div_wpr);
  const uint32_t k = fast_div(row, g.div_ny), j = row - k * (uint32_t)g.ny;
  const int x0 = 64 * (int)((uint32_t)w - row * (uint32_t)g.wpr);
  const float t1 = pl.pn[1] * ((pl.o[1] + pl.s[1] * (float)(int)j) - pl.po[1]);
  const float t2 = pl.pn[2] * ((pl.o[2] + pl.s[2] * (float)(int)k) - pl.po[2]);
  auto inside = [&](int x) -> bool {
    const float t0 = pl.pn[0] * ((pl.o[0] + pl.s[0] * (float)x) - pl.po[0]);
    return (t0 + t1) + t2 > g.iso;
  };
  const int n = min(64, g.nx - x0);
  const bool first = inside(x0), last = inside(x0 + n - 1);
  uint64_t m = first ? ~0ull : 0ull;
  if (first != last) {
    int lo = 0, hi = n - 1;  // inside(x0 + lo) == first, inside(x0 + hi) != first
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (inside(x0 + mid) == first)
        lo = mid;
      else
        hi = mid;
    }
    m = first ? low_mask(hi) : ~low_mask(hi);
  }
  bits[w] = m & low_mask(n);
}

// ---------------------------------------------------------------------------
// Tuning: per grid shape, the classify variant, scan sub-tiles and generate
// tile words.  Defaults are used until dax_hip_mc_autotune (or
// dax_hip_mc_set_tuning) records a choice for a shape.
// The classify variants are for rows of whole 64-point words; other rows are
// read as a flat stream, k_classify_flat.
struct Tuning {
  int cls_unroll = 4;   // words (vec 1) or 256-point chunks (vec 4) per wave
  int cls_vec = 4;      // floats per lane per load
  int scan_sub = 8;     // count tiles (waves) per count block
  int gen_tile = 512;   // generate tile words
  int gen_xcd = 0;      // 1: each XCD takes a contiguous range of generate tiles
};

std::mutex g_tune_mu;
Tuning g_tune_default;
bool g_tune_default_set = false;  // by a caller: it then holds for every size
std::map<std::tuple<int64_t, int64_t, int64_t>, Tuning> g_tune_cache;

// The launch shape of a volume without a choice of its own, while no caller has
// set the default.  Generate tiles: 64 words (spread over the waves
// launch_generate_src gives them) up to 2^20 words.  Beyond, tiles of 256 words
// can be dispatched in an order of their work, which pays where the surface
// takes few of the tiles (forward, 64 / 256 words: 256^3 points 59 / 65 us,
// 384^3 105 / 109, 512^3 194 / 176) and costs where most have output (dense
// 640^3 367 / 375, 1024^3 of 12.7 M vertices 1420 / 1435).  Which it is depends
// on the field, not on the shape, and the first gains more than the second
// loses; the autotuner times both.  A tile stages two rows beyond its own, so
// rows of more than 32 words take tiles of at least two rows.  Count blocks: one
// wave up to 2^16 words, to spread over more CUs (100 x 90 x 110 points: forward
// 37 / 38 / 40 us with 1 / 4 / 8 waves), four beyond (256^3: 68 / 67 / 69).
Tuning shape_tuning(int64_t nx, int64_t ny, int64_t nz) {
  Tuning t;
  const int64_t wpr = ceil_div(nx, 64), words = wpr * ny * nz;
  t.gen_tile = words <= (1 << 20) ? 64 : 256;
  while (t.gen_tile < 1024 && wpr > 32 && t.gen_tile < 2 * wpr) t.gen_tile *= 2;
  t.scan_sub = words <= (1 << 16) ? 1 : 4;
  return t;
}

Tuning tuning_for(int64_t nx, int64_t ny, int64_t nz) {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  auto it = g_tune_cache.find(std::make_tuple(nx, ny, nz));
  if (it != g_tune_cache.end()) return it->second;
  return g_tune_default_set ? g_tune_default : shape_tuning(nx, ny, nz);
}

bool valid_tuning(const Tuning& t) {
  const bool cls = (t.cls_vec == 1 && (t.cls_unroll == 8 || t.cls_unroll == 16 || t.cls_unroll == 32)) ||
                   (t.cls_vec == 4 && (t.cls_unroll == 2 || t.cls_unroll == 4 || t.cls_unroll == 8));
  const bool scan = t.scan_sub == 1 || t.scan_sub == 2 || t.scan_sub == 4 || t.scan_sub == 8;
  const bool gen = (t.gen_tile == 64 || t.gen_tile == 128 || t.gen_tile == 256 ||
                    t.gen_tile == 512 || t.gen_tile == 1024) &&
                   (t.gen_xcd == 0 || t.gen_xcd == 1);
  return cls && scan && gen;
}

// ---------------------------------------------------------------------------
// Per-cell outputs of the count step: case byte, NumFaces[case] and the
// exclusive triangle offset.  A wavefront takes kCellWords (8) consecutive
// row words: one load instruction brings all their neighbour words (lane
// 8u+v holds neighbour v of word u) and their bases, each word then reads its
// eight from the lanes and writes its 64 cells (lane = cell).  Words without
// a mixed cell need no case lookup, but testing every word for it keeps the
// words' chains from overlapping: where over a quarter of the neighbour words
// are mixed (rows of one word have half of them) all are looked up.  253x241x230
// (125 MB) of a sphere took 43 us with lookups only, 37 with tests only, this
// 38; 300^3 of noise 84, 87, 80.  Bound by the number of stores, 64 cells each
// wherever they start (3.3 TB/s); with scalar loads of the neighbours 78 us.
constexpr int kCellWords = 8;
__device__ __forceinline__ uint64_t readlane64(uint64_t v, int lane) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), lane);
  return (uint64_t)lo | ((uint64_t)hi << 32);
}

__global__ __launch_bounds__(256) void k_cell_outputs(VolGeom g, const uint64_t* __restrict__ bits,
                                                      CountSrc src, const Ctrl* __restrict__ ctrl,
                                                      uint8_t* __restrict__ cases,
                                                      int32_t* __restrict__ count,
                                                      int32_t* __restrict__ offsets) {
  __shared__ uint8_t s_nf[256];  // NumFaces per case
  s_nf[threadIdx.x] = (uint8_t)(c_case_table[threadIdx.x] >> 60);
  src.tpb_shift = (int)ctrl->tpb_shift;
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t w0 = ((int64_t)blockIdx.x * (256 / 64) + wv) * kCellWords;
  if (w0 >= g.nwords) return;  // wave-uniform
  const int64_t plane = (int64_t)g.wpr * g.ny;
  uint64_t mine = 0ull;  // neighbour (lane & 7) of word w0 + (lane >> 3)
  uint32_t base = 0u;    // triangle base of that word
  {
    const int64_t w = w0 + (lane >> 3);
    const int v = lane & 7;
    if (w < g.nwords) {
      const WordPos p = word_pos(g, w);
      if (p.has_y && p.has_z && (!(v & 1) || p.q + 1 < g.wpr))
        mine = bits[w + (v & 1) + ((v >> 1) & 1) * g.wpr + (v >> 2) * plane];
      if (offsets) base = (uint32_t)(word_bases(src, w) >> 32);
    }
  }
  const int64_t cx = g.nx - 1, cy = g.ny - 1;
  auto store_words = [&](auto look_up_all) {
#pragma unroll
    for (int u = 0; u < kCellWords; ++u) {
      const int64_t w = w0 + u;
      const WordPos p = word_pos(g, w < g.nwords ? w : w0);
      if (w >= g.nwords || !(p.has_y && p.has_z)) continue;  // wave-uniform: no cells
      uint64_t nb[8];
#pragma unroll
      for (int v = 0; v < 8; ++v) nb[v] = readlane64(mine, 8 * u + v);
      CellPlanes cp;
      cell_planes(p, nb[0], nb[1], nb[2], nb[3], nb[4], nb[5], nb[6], nb[7], cp);
      const bool valid = ((p.xmask >> lane) & 1ull) != 0;
      int cs = (nb[0] >> lane) & 1ull ? 255 : 0;  // no mixed corners: no faces
      uint32_t nf = 0u, incl = 0u;
      if (look_up_all.value || cp.active != 0ull) {  // wave-uniform
        cs = cell_case(cp, lane);
        nf = valid ? (uint32_t)s_nf[cs] : 0u;
        incl = offsets ? wave_incl_scan(nf) : 0u;
      }
      if (valid) {
        const int64_t cell = (int64_t)p.q * 64 + cx * (p.j + cy * (int64_t)p.k);
        const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)base, 8 * u);
        if (cases) (cases + cell)[lane] = (uint8_t)cs;
        if (count) (count + cell)[lane] = (int32_t)nf;
        if (offsets) (offsets + cell)[lane] = (int32_t)(first + incl - nf);
      }
    }
  };
  if (__popcll(__ballot(mine != 0ull && mine != ~0ull)) > 16)
    store_words(std::true_type{});
  else
    store_words(std::false_type{});
}

__global__ void k_interpolate_scalar(const float* __restrict__ in, const int32_t* __restrict__ first,
                                     const int32_t* __restrict__ second,
                                     const float* __restrict__ weight, int64_t n,
                                     float* __restrict__ out) {
  const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= n) return;
  const float a = in[first[u]], b = in[second[u]];
  out[u] = a + weight[u] * (b - a);
}

__global__ void k_interpolate_vec3(const float* __restrict__ in, const int32_t* __restrict__ first,
                                   const int32_t* __restrict__ second,
                                   const float* __restrict__ weight, int64_t n,
                                   float* __restrict__ out) {
  const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= n) return;
  const int64_t a = 3 * (int64_t)first[u], b = 3 * (int64_t)second[u];
  const float w = weight[u];
#pragma unroll
  for (int d = 0; d < 3; ++d) out[3 * u + d] = in[a + d] + w * (in[b + d] - in[a + d]);
}

// A block's 256 vectors of three, from entry `first` of n on, through LDS: 192
// 16-byte stores instead of three 4-byte ones a thread at a stride of 12
// (s: 768 floats).
__device__ __forceinline__ void store_block3(float* __restrict__ out, int64_t first, int64_t n,
                                             const float v[3], f32x4* s) {
  const int tid = threadIdx.x;
  float* sf = reinterpret_cast<float*>(s);
#pragma unroll
  for (int d = 0; d < 3; ++d) sf[3 * tid + d] = v[d];
  __syncthreads();
  float* o = out + 3 * first;
  const int m = 3 * (int)min((int64_t)256, n - first);
  if ((reinterpret_cast<uintptr_t>(o) & 15u) == 0) {
    if (4 * tid + 4 <= m)
      reinterpret_cast<f32x4*>(o)[tid] = s[tid];
    else
      for (int i = 4 * tid; i < m; ++i) o[i] = sf[i];
  } else {
    for (int i = tid; i < m; i += 256) o[i] = sf[i];
  }
}

// A plane of the gradient kernels fills its blocks of 256 to three quarters or
// more: blocks march over planes.  Below that a thread takes one point (cell)
// of the flat index, so that small planes leave no lanes idle and no grid more
// blocks than a launch takes (point gradient, flat / marching: 8 x 8 x 500000
// 131 / 282 us, 4 x 4 x 1000000 44 / 417, 300 x 1 x 100000 123 / 166, 17 x 13 x
// 50000 39 / 35, 16 x 16 x 100000 104 / 99).
inline bool march_planes(int64_t plane) { return 4 * plane >= 3 * 256 * ceil_div(plane, 256); }

// Planes a block of the gradient kernels marches through: neighbours in z stay
// in registers and indexes are formed once, up to 8 where that leaves enough
// blocks.
inline int gradient_planes(int64_t plane_blocks, int64_t nz) {
  return (int)std::max<int64_t>(1, std::min<int64_t>(8, plane_blocks * nz / 4096));
}

// A block takes 256 points of a plane and the points above them in `planes`
// planes.  Blocks of one XCD are next to each other, so that the rows around a
// point are in its L2.  Bound by the stores (12 of the 16 bytes a point moves).
// Again and again on one field, 253x241x230: 66 us with one plane a block, 55
// with eight, 39 in XCD order; 512^3: 746, 521, 506 (4.2 TB/s).
__global__ __launch_bounds__(256) void k_point_gradient(VolGeom g, int planes, FastDiv div_pb,
                                                        const float* __restrict__ f,
                                                        float* __restrict__ grad) {
  __shared__ f32x4 s[2][192];
  const int32_t plane = g.nx * g.ny;
  const uint32_t id = (uint32_t)xcd_tile_runs(blockIdx.x, gridDim.x), zc = fast_div(id, div_pb);
  const int32_t first = (int32_t)(id - zc * (uint32_t)ceil_div((int64_t)plane, 256)) * 256;
  const int z0 = (int)zc * planes, z1 = min(z0 + planes, g.nz);
  const uint32_t p = (uint32_t)min(first + (int32_t)threadIdx.x, plane - 1);
  const int y = (int)fast_div(p, g.div_nx), x = (int)(p - (uint32_t)y * (uint32_t)g.nx);
  const int xm = x > 0 ? -1 : 0, xp = x + 1 < g.nx ? 1 : 0;
  const int ym = y > 0 ? -g.nx : 0, yp = y + 1 < g.ny ? g.nx : 0;
  const float* q = f + (int64_t)z0 * plane + p;
  float c = q[0], before = z0 > 0 ? q[-(int64_t)plane] : c;
  for (int z = z0; z < z1; ++z, q += plane) {
    const float after = z + 1 < g.nz ? q[plane] : c;
    const float lo[3] = {q[xm], q[ym], before}, hi[3] = {q[xp], q[yp], after};
    float gr[3];
    gradient_finish(g, x, y, z, lo, hi, gr);
    store_block3(grad + 3 * (int64_t)z * plane, first, plane, gr, s[(z - z0) & 1]);
    before = c;
    c = after;
  }
}

// The same for planes that would leave a marching block idle, a thread per point
// of the flat index (its stores through LDS took as long).
__global__ __launch_bounds__(256) void k_point_gradient_flat(VolGeom g, int64_t n,
                                                             const float* __restrict__ f,
                                                             float* __restrict__ grad) {
  const int64_t at = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (at >= n) return;
  const uint32_t p = (uint32_t)at;
  const uint32_t row = fast_div(p, g.div_nx), z = fast_div(row, g.div_ny);
  float gr[3];
  point_gradient(g, FieldArray{f}, (int)(p - row * (uint32_t)g.nx),
                 (int)(row - z * (uint32_t)g.ny), (int)z, gr);
  store3(grad + 3 * at, gr[0], gr[1], gr[2]);
}

// Gradient of the cell (i, j, z) from a quarter of its corners' values, lower
// and upper plane (the weights are +-0.25; the product with either sign rounds
// alike): CellGradient (dax/worklet/CellGradient.h:28-48), weights of
// DerivativeWeights(Voxel) at the centre in the corner order of
// TopologyUniform.h:139-159; sum in vertex order, divided by the voxel width
// coords[6]-coords[0] (Derivative.h:37-75).
__device__ __forceinline__ float cell_width(const VolGeom& g, int d, int n) {
  const float a = g.origin[d] + g.spacing[d] * (float)n;
  const float b = g.origin[d] + g.spacing[d] * (float)(n + 1);
  return b - a;
}
__device__ __forceinline__ void cell_gradient(const float lo[4], const float hi[4],
                                              const float width[3], float gr[3]) {
  float s[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int v = 0; v < 8; ++v) {
    const float t = v < 4 ? lo[v & 3] : hi[v & 3];
    const bool px = (v & 3) == 1 || (v & 3) == 2, py = (v & 2) != 0, pz = v >= 4;
    s[0] = px ? s[0] + t : s[0] - t;
    s[1] = py ? s[1] + t : s[1] - t;
    s[2] = pz ? s[2] + t : s[2] - t;
  }
  // s / w; a power of two divides exactly by its reciprocal
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const uint32_t u = __float_as_uint(width[d]);
    const bool pow2 = (u & 0x7fffffu) == 0u && (u >> 23) - 1u < 253u;
    gr[d] = !__ballot(!pow2) ? s[d] * __uint_as_float(0x7f000000u - u) : s[d] / width[d];
  }
}

// Blocks as k_point_gradient's; 253x241x230: 64, 47, 41 us, 512^3: 829, 523,
// 493 (a thread per cell with 64-bit divisions and stores at a stride of 12
// bytes, among other work: 85 us where this takes 57..66).
__global__ __launch_bounds__(256) void k_cell_gradient(VolGeom g, int planes, FastDiv div_pb,
                                                       FastDiv div_cx,
                                                       const float* __restrict__ f,
                                                       float* __restrict__ out) {
  __shared__ f32x4 s[2][192];
  const int32_t cx = g.nx - 1, cy = g.ny - 1, cz = g.nz - 1, cells = cx * cy;  // of a plane
  const int32_t plane = g.nx * g.ny;
  const uint32_t id = (uint32_t)xcd_tile_runs(blockIdx.x, gridDim.x), zc = fast_div(id, div_pb);
  const int32_t first = (int32_t)(id - zc * (uint32_t)ceil_div((int64_t)cells, 256)) * 256;
  const int z0 = (int)zc * planes, z1 = min(z0 + planes, cz);
  const uint32_t c = (uint32_t)min(first + (int32_t)threadIdx.x, cells - 1);
  const int j = (int)fast_div(c, div_cx), i = (int)(c - (uint32_t)j * (uint32_t)cx);
  float width[3] = {cell_width(g, 0, i), cell_width(g, 1, j), 0.0f};
  const float* q = f + (int64_t)z0 * plane + i + (int64_t)j * g.nx;
  float lo[4] = {0.25f * q[0], 0.25f * q[1], 0.25f * q[g.nx + 1], 0.25f * q[g.nx]};
  for (int z = z0; z < z1; ++z) {
    q += plane;
    const float hi[4] = {0.25f * q[0], 0.25f * q[1], 0.25f * q[g.nx + 1], 0.25f * q[g.nx]};
    width[2] = cell_width(g, 2, z);
    float gr[3];
    cell_gradient(lo, hi, width, gr);
    store_block3(out + 3 * (int64_t)z * cells, first, cells, gr, s[(z - z0) & 1]);
#pragma unroll
    for (int v = 0; v < 4; ++v) lo[v] = hi[v];
  }
}

__global__ __launch_bounds__(256) void k_cell_gradient_flat(VolGeom g, int64_t n, FastDiv div_cx,
                                                            FastDiv div_cy,
                                                            const float* __restrict__ f,
                                                            float* __restrict__ out) {
  const int64_t at = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (at >= n) return;
  const uint32_t c = (uint32_t)at;
  const uint32_t row = fast_div(c, div_cx), z = fast_div(row, div_cy);
  const int i = (int)(c - row * (uint32_t)(g.nx - 1)), j = (int)(row - z * (uint32_t)(g.ny - 1));
  const float* q = f + i + (int64_t)g.nx * (j + (int64_t)g.ny * z);
  const float* u = q + (int64_t)g.nx * g.ny;
  const float lo[4] = {0.25f * q[0], 0.25f * q[1], 0.25f * q[g.nx + 1], 0.25f * q[g.nx]};
  const float hi[4] = {0.25f * u[0], 0.25f * u[1], 0.25f * u[g.nx + 1], 0.25f * u[g.nx]};
  const float width[3] = {cell_width(g, 0, i), cell_width(g, 1, j), cell_width(g, 2, (int)z)};
  float gr[3];
  cell_gradient(lo, hi, width, gr);
  store3(out + 3 * at, gr[0], gr[1], gr[2]);
}

}  // namespace mc
}  // namespace daxhip

// ---------------------------------------------------------------------------
// C-ABI
using namespace daxhip;
using namespace daxhip::mc;

namespace {

int make_geom(int64_t nx, int64_t ny, int64_t nz, const float* origin, const float* spacing,
              float iso, VolGeom& g) {
  if (nx < 1 || ny < 1 || nz < 1) {
    set_error("dax_hip_mc: grid dimensions must be >= 1 (got %lld x %lld x %lld)", (long long)nx,
              (long long)ny, (long long)nz);
    return DAX_HIP_BAD_VALUE;
  }
  if (nx * ny * nz > 0x7fffffffLL) {
    set_error("dax_hip_mc: %lld points exceed the int32 dax::Id range",
              (long long)(nx * ny * nz));
    return DAX_HIP_BAD_VALUE;
  }
  if (ceil_div(nx, 64) > kMaxWpr) {
    set_error("dax_hip_mc: nx=%lld exceeds the supported row length %d", (long long)nx,
              kMaxWpr * 64);
    return DAX_HIP_BAD_VALUE;
  }
  g.nx = (int32_t)nx;
  g.ny = (int32_t)ny;
  g.nz = (int32_t)nz;
  g.wpr = (int32_t)ceil_div(nx, 64);
  g.iso = iso;
  for (int d = 0; d < 3; ++d) {
    g.origin[d] = origin ? origin[d] : 0.0f;
    g.spacing[d] = spacing ? spacing[d] : 1.0f;
  }
  g.field_off = 0;
  g.word_off = 0;
  g.nwords = (int64_t)g.wpr * ny * nz;
  g.tile_off = 0;
  set_geom_divs(g);
  return DAX_HIP_OK;
}

// Geometry and plane of a slice; the isovalue is dot(normal, origin) summed
// from component 0 (dax/worklet/Slice.h:44,104; dax/Types.h:611-621).
int make_slice(int64_t nx, int64_t ny, int64_t nz, const float* origin, const float* spacing,
               const float* plane_origin, const float* plane_normal, VolGeom& g,
               FieldPlane& pl) {
  if (!plane_origin || !plane_normal) {
    set_error("dax_hip_mc_slice: plane origin and normal are required");
    return DAX_HIP_BAD_VALUE;
  }
  float iso = plane_normal[0] * plane_origin[0];
  iso += plane_normal[1] * plane_origin[1];
  iso += plane_normal[2] * plane_origin[2];
  const int rc = make_geom(nx, ny, nz, origin, spacing, iso, g);
  if (rc) return rc;
  for (int d = 0; d < 3; ++d) {
    pl.o[d] = g.origin[d];
    pl.s[d] = g.spacing[d];
    pl.po[d] = plane_origin[d];
    pl.pn[d] = plane_normal[d];
  }
  return DAX_HIP_OK;
}

int check_ws(const VolGeom& g, size_t ws_bytes, Workspace& L, void* ws) {
  L = workspace_layout(g.nwords);
  if (!ws || ws_bytes < L.bytes) {
    set_error("dax_hip_mc: workspace of %zu bytes is smaller than the %zu needed", ws_bytes,
              L.bytes);
    return DAX_HIP_BAD_VALUE;
  }
  return DAX_HIP_OK;
}

// Classify the whole volume.
int launch_bits(const VolGeom& g, const float* field, char* ws, const Workspace& L,
                const Tuning& tu, hipStream_t s) {
  uint64_t* bits = (uint64_t*)(ws + L.off_bits);
  const bool aligned = (g.nx % 64) == 0 && (g.field_off % 4) == 0 && ((uintptr_t)field % 16) == 0;
  if (!aligned) {
    // 8192 points, 8 float4 loads per thread, for rows of full or half words;
    // shorter rows hold fewer points per word, so four times the words
    const int tw = g.nx > 32 ? 128 : 512;
    const dim3 grid((unsigned)ceil_div(g.nwords, tw)), block(256);
    if (tw == 128)
      k_classify_flat<128><<<grid, block, 0, s>>>(g, field, bits, g.nwords);
    else
      k_classify_flat<512><<<grid, block, 0, s>>>(g, field, bits, g.nwords);
    DAXHIP_LAUNCH_CHECK("k_classify_flat");
    return DAX_HIP_OK;
  }
  const int vec = tu.cls_vec, unroll = tu.cls_unroll;
  const int64_t units = vec == 4 ? ceil_div(g.nwords, 4) : g.nwords;  // chunks or words
  const int64_t waves = ceil_div(units, unroll);
  const dim3 grid((unsigned)ceil_div(waves * 64, 256)), block(256);
#define DAXHIP_CLS(U) k_classify<U><<<grid, block, 0, s>>>(g, field, bits, g.nwords)
#define DAXHIP_CLS4(U) k_classify_v4<U><<<grid, block, 0, s>>>(g, field, bits, g.nwords)
  if (vec == 4) {
    if (unroll == 2) DAXHIP_CLS4(2);
    else if (unroll == 4) DAXHIP_CLS4(4);
    else DAXHIP_CLS4(8);
  } else {
    if (unroll == 8) DAXHIP_CLS(8);
    else if (unroll == 32) DAXHIP_CLS(32);
    else DAXHIP_CLS(16);
  }
#undef DAXHIP_CLS
#undef DAXHIP_CLS4
  DAXHIP_LAUNCH_CHECK("k_classify");
  return DAX_HIP_OK;
}

// Generate tile words of a tuning (launch_generate_src's dispatch).
int gen_tile_words(const Tuning& tu) {
  return (tu.gen_tile == 64 || tu.gen_tile == 128 || tu.gen_tile == 256 || tu.gen_tile == 1024)
             ? tu.gen_tile
             : 512;
}

// A count block holds two count tiles per wave, with the waves of
// launch_scan's dispatch (1, 2, 8, else 4).
int tiles_per_block_shift(const Tuning& tu) {
  return tu.scan_sub == 1 ? 1 : (tu.scan_sub == 2 ? 2 : (tu.scan_sub == 8 ? 4 : 3));
}

// Where the word bases come from (the tiles per count block
// come from the control block: the scan may have run under another tuning).
CountSrc count_src(const char* ws, const Workspace& L) {
  return CountSrc{(const uint32_t*)(ws + L.off_counts),
                  (const unsigned long long*)(ws + L.off_tsum),
                  (const unsigned long long*)(ws + L.off_tpre), L.n_ctiles, 0, 0};
}

// Count + block-sum scan over the whole volume (scan_sub waves, i.e.
// 2 * scan_sub count tiles, per count block).
int launch_scan(const VolGeom& g, char* ws, const Workspace& L, const Tuning& tu, hipStream_t s,
                ScanOut so = ScanOut{nullptr, nullptr}) {
  const uint64_t* bits = (const uint64_t*)(ws + L.off_bits);
  uint32_t* lpre = (uint32_t*)(ws + L.off_counts);
  unsigned long long* tloc = (unsigned long long*)(ws + L.off_tsum);
  unsigned long long* bsum = (unsigned long long*)(ws + L.off_bsum);
  unsigned long long* bpre = (unsigned long long*)(ws + L.off_tpre);
  const int64_t n = L.n_ctiles;
  const int waves = tu.scan_sub;
  // generate classes when a count block covers whole generate tiles
  const int tw = gen_tile_words(tu);
  const int block_words = 2 * (waves == 1 || waves == 2 || waves == 8 ? waves : 4) * kCountTile;
  const TileClasses tc{(uint8_t*)(ws + L.off_gcls),
                       tw >= kCountTile && tw <= block_words ? tw : 0};
  const int64_t nblocks = ceil_div(n, 2 * waves);
  if (nblocks > 0) {
    const dim3 grid((unsigned)nblocks), block(64 * waves);
    switch (waves) {
      case 1: k_count<1><<<grid, block, 0, s>>>(g, bits, lpre, tloc, bsum, tc, n); break;
      case 2: k_count<2><<<grid, block, 0, s>>>(g, bits, lpre, tloc, bsum, tc, n); break;
      case 8: k_count<8><<<grid, block, 0, s>>>(g, bits, lpre, tloc, bsum, tc, n); break;
      default: k_count<4><<<grid, block, 0, s>>>(g, bits, lpre, tloc, bsum, tc, n); break;
    }
    DAXHIP_LAUNCH_CHECK("k_count");
  }
  // with the dispatch order of the generate tiles, in units of two tiles a
  // plane apart when tiles split planes evenly and the units fill groups of 8
  const int64_t ng = ceil_div(g.nwords, (int64_t)tw);
  const int64_t plane = (int64_t)g.wpr * g.ny;
  const int64_t sp = plane % tw == 0 ? plane / tw : 0;
  constexpr int64_t kUnitG = kOrderUnitTiles;
  const bool units = tc.tw > 0 && sp > 0 && ng % (kUnitG * sp) == 0 && (ng / kUnitG) % 8 == 0 &&
                     ceil_div(ng / kUnitG, (int64_t)kTsumThreads) * kUnitG <= kOrderRegTiles;
  const GenOrder go{tc.gcls, g.nwords, tw, tc.tw > 0, units ? (uint32_t)sp : 0u,
                    (uint32_t*)(ws + L.off_order)};
  if (ceil_div(ceil_div(g.nwords, (int64_t)tw), (int64_t)kTsumThreads) > kOrderRegTiles)
    k_scan_tsums<true><<<1, dim3(kTsumThreads), 0, s>>>(
        bsum, bpre, nblocks, tloc, n, (Ctrl*)(ws + L.off_ctrl), go, tiles_per_block_shift(tu), so);
  else
    k_scan_tsums<false><<<1, dim3(kTsumThreads), 0, s>>>(
        bsum, bpre, nblocks, tloc, n, (Ctrl*)(ws + L.off_ctrl), go, tiles_per_block_shift(tu), so);
  DAXHIP_LAUNCH_CHECK("k_scan_tsums");
  return DAX_HIP_OK;
}

// Generate tiles of TW words [t_lo, t_hi) (all when t_hi < 0).
template <int TW, int NT, class Src>
int launch_generate_tw(const VolGeom& g, const Src& field, const char* ws, const Workspace& L,
                       unsigned flags, const OutPtrs& o, int64_t cap_points, int64_t cap_tris,
                       int64_t* counts, const Tuning& tu, hipStream_t s, int64_t t_lo,
                       int64_t t_hi) {
  const int xcd = tu.gen_xcd;
  const size_t lds = GenLayout<TW, NT>(g.wpr).bytes();
  const int64_t all = ceil_div(g.nwords, (int64_t)TW);
  if (t_hi < 0) t_hi = all;
  const int64_t ntiles = std::max<int64_t>(t_hi - t_lo, 1);
  const CountSrc cs = count_src(ws, L);
  // the order lists tiles of at least a count tile: it has no entries for more
  const uint32_t* order = TW >= kCountTile && t_lo == 0 && t_hi == all
                              ? (const uint32_t*)(ws + L.off_order) : nullptr;
#define DAXHIP_GEN(DEDUP)                                                                        \
  k_generate<TW, NT, Src, DEDUP><<<dim3((unsigned)ntiles), dim3(NT), lds, s>>>(                  \
      g, field, (const uint64_t*)(ws + L.off_bits), cs, (const Ctrl*)(ws + L.off_ctrl), o, flags, \
      cap_points, cap_tris, counts, xcd, t_lo, ntiles, order)
  if (flags & DAX_HIP_MC_DEDUP)
    DAXHIP_GEN(true);
  else
    DAXHIP_GEN(false);
#undef DAXHIP_GEN
  DAXHIP_LAUNCH_CHECK("k_generate");
  return DAX_HIP_OK;
}

template <class Src>
int launch_generate_src(const VolGeom& g, const Src& field, const char* ws, const Workspace& L,
                        unsigned flags, const OutPtrs& o, int64_t cap_points, int64_t cap_tris,
                        int64_t* counts, const Tuning& tu, hipStream_t s, int64_t t_lo = 0,
                        int64_t t_hi = -1) {
#define DAXHIP_GEN_TW(TW, NT)                                                                  \
  launch_generate_tw<TW, NT>(g, field, ws, L, flags, o, cap_points, cap_tris, counts, tu, s, t_lo, \
                             t_hi)
  switch (tu.gen_tile) {
    case 64:
      // A wave per tile runs its rounds one after another, so few tiles leave
      // the chip waiting on chains: four waves share a tile's outputs up to
      // 2^18 words, two up to 2^20 (128^3 points: 43 / 28 / 18 us with one /
      // two / four waves, 256^3 47 / 39 / 39, 384^3 58 / 56 / 67, 512^3 84 /
      // 105 / 155).
      if (g.nwords <= (1 << 18)) return DAXHIP_GEN_TW(64, 256);
      if (g.nwords <= (1 << 20)) return DAXHIP_GEN_TW(64, 128);
      return DAXHIP_GEN_TW(64, 64);
    case 128:
      return DAXHIP_GEN_TW(128, 128);
    case 256:
      return DAXHIP_GEN_TW(256, 256);
    case 1024:
      return DAXHIP_GEN_TW(1024, 1024);
    default:
      return DAXHIP_GEN_TW(512, 512);
  }
#undef DAXHIP_GEN_TW
}

int launch_generate(const VolGeom& g, const float* field, const char* ws, const Workspace& L,
                    unsigned flags, const OutPtrs& o, int64_t cap_points, int64_t cap_tris,
                    int64_t* counts, const Tuning& tu, hipStream_t s, int64_t t_lo = 0,
                    int64_t t_hi = -1) {
  return launch_generate_src(g, FieldArray{field + g.field_off}, ws, L, flags, o, cap_points,
                             cap_tris, counts, tu, s, t_lo, t_hi);
}

// Slice classify over the whole volume.
int launch_bits_plane(const VolGeom& g, const FieldPlane& pl, char* ws, const Workspace& L,
                      hipStream_t s) {
  k_classify_plane<<<dim3((unsigned)ceil_div(g.nwords, 256)), dim3(256), 0, s>>>(
      g, pl, (uint64_t*)(ws + L.off_bits));
  DAXHIP_LAUNCH_CHECK("k_classify_plane");
  return DAX_HIP_OK;
}

// The kernels of a forward over the whole volume.
int launch_forward(const VolGeom& g, const float* field, char* ws, const Workspace& L,
                   unsigned flags, const OutPtrs& o, int64_t cap_points, int64_t cap_tris,
                   int64_t* counts, const Tuning& tu, hipStream_t s) {
  int rc;
  if ((rc = launch_bits(g, field, ws, L, tu, s))) return rc;
  if ((rc = launch_scan(g, ws, L, tu, s))) return rc;
  return launch_generate(g, field, ws, L, flags, o, cap_points, cap_tris, counts, tu, s);
}

int check_outputs(const VolGeom& g, const float* field, unsigned flags, const float* vertices,
                  const int32_t* conn, const uint32_t* edges, const int64_t* counts) {
  if (!field || !vertices || !conn || !counts) {
    set_error("dax_hip_mc: field, vertices, connectivity and counts are required");
    return DAX_HIP_BAD_VALUE;
  }
  if (edges && (!(flags & DAX_HIP_MC_DEDUP) || (int64_t)g.nx * g.ny * g.nz > (1LL << 30))) {
    set_error("dax_hip_mc: the compact edge list needs dedup and at most 2^30 points");
    return DAX_HIP_BAD_VALUE;
  }
  return DAX_HIP_OK;
}

// T and U within the int32 dax::Id range.
int check_totals(int64_t t, int64_t u) {
  if (u > 0x7fffffffLL || 3 * t > 0x7fffffffLL) {
    set_error("dax_hip_mc: %lld triangles / %lld points exceed the int32 dax::Id range",
              (long long)t, (long long)u);
    return DAX_HIP_EXEC_ERROR;
  }
  return DAX_HIP_OK;
}

// Count + scan of classified bits, with {T, U} read back (synchronous).
int count_sync(const VolGeom& g, char* ws, const Workspace& L, const Tuning& tu, int64_t* h_tris,
               int64_t* h_points, hipStream_t s) {
  int64_t c[2] = {0, 0};
  HostSlot slot(s);
  int rc;
  if ((rc = launch_scan(g, ws, L, tu, s, ScanOut{nullptr, slot.p}))) return rc;
  unsigned long long vt[2];
  if (!slot.p)
    DAXHIP_CHECK(hipMemcpyAsync(vt, ws + L.off_ctrl + offsetof(Ctrl, total_v), sizeof(vt),
                                hipMemcpyDeviceToHost, s));
  DAXHIP_CHECK(slot.wait());
  c[0] = slot.p ? ((volatile int64_t*)slot.p)[0] : (int64_t)vt[1];
  c[1] = slot.p ? ((volatile int64_t*)slot.p)[1] : (int64_t)vt[0];
  *h_tris = c[0];
  *h_points = c[1];
  return check_totals(c[0], c[1]);
}

}  // namespace

extern "C" {

size_t dax_hip_mc_workspace_bytes(int64_t nx, int64_t ny, int64_t nz) {
  if (nx < 1 || ny < 1 || nz < 1) return 0;
  return workspace_layout(ceil_div(nx, 64) * ny * nz).bytes;
}

int dax_hip_mc_bits(const float* d_field, int64_t nx, int64_t ny, int64_t nz, float iso,
                    void* d_workspace, size_t workspace_bytes, void* stream) {
  VolGeom g;
  int rc = make_geom(nx, ny, nz, nullptr, nullptr, iso, g);
  if (rc) return rc;
  Workspace L;
  if ((rc = check_ws(g, workspace_bytes, L, d_workspace))) return rc;
  if (!d_field) {
    set_error("dax_hip_mc_bits: field is NULL");
    return DAX_HIP_BAD_VALUE;
  }
  return launch_bits(g, d_field, (char*)d_workspace, L, tuning_for(nx, ny, nz),
                     (hipStream_t)stream);
}

int dax_hip_mc_scan(int64_t nx, int64_t ny, int64_t nz, void* d_workspace, size_t workspace_bytes,
                    void* stream) {
  VolGeom g;
  int rc = make_geom(nx, ny, nz, nullptr, nullptr, 0.0f, g);
  if (rc) return rc;
  Workspace L;
  if ((rc = check_ws(g, workspace_bytes, L, d_workspace))) return rc;
  return launch_scan(g, (char*)d_workspace, L, tuning_for(nx, ny, nz), (hipStream_t)stream);
}

int dax_hip_mc_generate(const float* d_field, int64_t nx, int64_t ny, int64_t nz,
                        const float* h_origin3, const float* h_spacing3, float iso,
                        unsigned flags, const void* d_workspace, size_t workspace_bytes,
                        float* d_vertices, float* d_normals, int32_t* d_conn, uint32_t* d_edges,
                        int32_t* d_interp_first, int32_t* d_interp_second,
                        float* d_interp_weight, int64_t cap_points, int64_t cap_tris,
                        int64_t* d_counts, void* stream) {
  VolGeom g;
  int rc = make_geom(nx, ny, nz, h_origin3, h_spacing3, iso, g);
  if (rc) return rc;
  Workspace L;
  if ((rc = check_ws(g, workspace_bytes, L, (void*)d_workspace))) return rc;
  if ((rc = check_outputs(g, d_field, flags, d_vertices, d_conn, d_edges, d_counts))) return rc;
  OutPtrs o{d_vertices, d_normals, d_conn, d_edges, d_interp_first, d_interp_second,
            d_interp_weight};
  return launch_generate(g, d_field, (const char*)d_workspace, L, flags, o, cap_points, cap_tris,
                         d_counts, tuning_for(nx, ny, nz), (hipStream_t)stream);
}

int dax_hip_mc_classify(const float* d_field, int64_t nx, int64_t ny, int64_t nz, float iso,
                        void* d_workspace, size_t workspace_bytes, int64_t* d_counts,
                        void* stream) {
  VolGeom g;
  int rc = make_geom(nx, ny, nz, nullptr, nullptr, iso, g);
  if (rc) return rc;
  Workspace L;
  if ((rc = check_ws(g, workspace_bytes, L, d_workspace))) return rc;
  if (!d_field) {
    set_error("dax_hip_mc_classify: field is NULL");
    return DAX_HIP_BAD_VALUE;
  }
  hipStream_t s = (hipStream_t)stream;
  char* ws = (char*)d_workspace;
  const Tuning tu = tuning_for(nx, ny, nz);
  if ((rc = launch_bits(g, d_field, ws, L, tu, s))) return rc;
  return launch_scan(g, ws, L, tu, s, ScanOut{d_counts, nullptr});
}

int dax_hip_mc_count(const float* d_field, int64_t nx, int64_t ny, int64_t nz, float iso,
                     void* d_workspace, size_t workspace_bytes, int64_t* h_tris,
                     int64_t* h_points, void* stream) {
  VolGeom g;
  int rc = make_geom(nx, ny, nz, nullptr, nullptr, iso, g);
  if (rc) return rc;
  Workspace L;
  if ((rc = check_ws(g, workspace_bytes, L, d_workspace))) return rc;
  if (!d_field || !h_tris || !h_points) {
    set_error("dax_hip_mc_count: field, h_tris and h_points are required");
    return DAX_HIP_BAD_VALUE;
  }
  hipStream_t s = (hipStream_t)stream;
  const Tuning tu = tuning_for(nx, ny, nz);
  if ((rc = launch_bits(g, d_field, (char*)d_workspace, L, tu, s))) return rc;
  return count_sync(g, (char*)d_workspace, L, tu, h_tris, h_points, s);
}

int dax_hip_mc_forward(const float* d_field, int64_t nx, int64_t ny, int64_t nz,
                       const float* h_origin3, const float* h_spacing3, float iso,
                       unsigned flags, void* d_workspace, size_t workspace_bytes,
                       float* d_vertices, float* d_normals, int32_t* d_conn, uint32_t* d_edges,
                       int32_t* d_interp_first, int32_t* d_interp_second,
                       float* d_interp_weight, int64_t cap_points, int64_t cap_tris,
                       int64_t* d_counts, void* stream) {
  VolGeom g;
  int rc = make_geom(nx, ny, nz, h_origin3, h_spacing3, iso, g);
  if (rc) return rc;
  Workspace L;
  if ((rc = check_ws(g, workspace_bytes, L, d_workspace))) return rc;
  if ((rc = check_outputs(g, d_field, flags, d_vertices, d_conn, d_edges, d_counts))) return rc;
  hipStream_t s = (hipStream_t)stream;
  char* ws = (char*)d_workspace;
  const Tuning tu = tuning_for(nx, ny, nz);
  OutPtrs o{d_vertices, d_normals, d_conn, d_edges, d_interp_first, d_interp_second,
            d_interp_weight};
  return launch_forward(g, d_field, ws, L, flags, o, cap_points, cap_tris, d_counts, tu, s);
}

// ---- forward without allocation -------------------------------------------
// dax_hip_mc_forward with its workspace in a file-scope device array, for
// callers that cannot allocate (code under graph capture, serving loops):
// grids of up to kNoAllocMaxWords row words (512^3 points have 2^21).  Every GPU
// the library runs on holds the array until the process ends.  Calls that
// overlap on one GPU share the array and race.
constexpr int64_t kNoAllocMaxWords = 2484927;
constexpr size_t kNoAllocScratchBytes = (size_t)32 << 20;  // 12.3 bytes a word
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {
constexpr int kNoAllocDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kNoAllocDevices] = {};  // device address of `scratch`, per device

// The current device's copy of `scratch`, looked up once per device (with
// that device current); host code uses this address, never the array's name.
int scratch_on_device(void** ptr) {
  int dev = 0;
  DAXHIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kNoAllocDevices) {
    set_error("dax_hip_mc_forward_noalloc: device %d beyond the scratch table", dev);
    return DAX_HIP_BAD_VALUE;
  }
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) return check_hip(e != hipSuccess ? e : hipErrorInvalidSymbol,
                                                "hipGetSymbolAddress(scratch)");
    g_scratch_ptr[dev] = p;
  }
  *ptr = g_scratch_ptr[dev];
  return DAX_HIP_OK;
}
}  // namespace

int dax_hip_mc_forward_noalloc(const float* d_field, int64_t nx, int64_t ny, int64_t nz,
                               const float* h_origin3, const float* h_spacing3, float iso,
                               unsigned flags, float* d_vertices, float* d_normals,
                               int32_t* d_conn, uint32_t* d_edges, int32_t* d_interp_first,
                               int32_t* d_interp_second, float* d_interp_weight,
                               int64_t cap_points, int64_t cap_tris, int64_t* d_counts,
                               void* stream) {
  VolGeom g;
  int rc = make_geom(nx, ny, nz, h_origin3, h_spacing3, iso, g);
  if (rc) return rc;
  const Workspace L = workspace_layout(g.nwords);
  if (g.nwords > kNoAllocMaxWords || L.fwd_bytes > kNoAllocScratchBytes) {
    set_error("dax_hip_mc_forward_noalloc: a %lld x %lld x %lld grid needs %zu bytes of scratch "
              "(%lld row words), there is room for %lld row words",
              (long long)nx, (long long)ny, (long long)nz, L.fwd_bytes, (long long)g.nwords,
              (long long)kNoAllocMaxWords);
    return DAX_HIP_BAD_VALUE;
  }
  if ((rc = check_outputs(g, d_field, flags, d_vertices, d_conn, d_edges, d_counts))) return rc;
  void* ws = nullptr;
  if ((rc = scratch_on_device(&ws))) return rc;
  OutPtrs o{d_vertices, d_normals, d_conn, d_edges, d_interp_first, d_interp_second,
            d_interp_weight};
  return launch_forward(g, d_field, (char*)ws, L, flags, o, cap_points, cap_tris, d_counts,
                        tuning_for(nx, ny, nz), (hipStream_t)stream);
}

// ---- slice: marching cubes of the plane distance, computed in the kernels
// (SliceCount / SliceGenerate, dax/worklet/Slice.h:28-173, on a uniform
// grid; no field in memory).
int dax_hip_mc_slice_classify(int64_t nx, int64_t ny, int64_t nz, const float* h_origin3,
                              const float* h_spacing3, const float* h_plane_origin3,
                              const float* h_plane_normal3, void* d_workspace,
                              size_t workspace_bytes, int64_t* d_counts, void* stream) {
  VolGeom g;
  FieldPlane pl;
  int rc = make_slice(nx, ny, nz, h_origin3, h_spacing3, h_plane_origin3, h_plane_normal3, g, pl);
  if (rc) return rc;
  Workspace L;
  if ((rc = check_ws(g, workspace_bytes, L, d_workspace))) return rc;
  hipStream_t s = (hipStream_t)stream;
  char* ws = (char*)d_workspace;
  if ((rc = launch_bits_plane(g, pl, ws, L, s))) return rc;
  return launch_scan(g, ws, L, tuning_for(nx, ny, nz), s, ScanOut{d_counts, nullptr});
}

int dax_hip_mc_slice_count(int64_t nx, int64_t ny, int64_t nz, const float* h_origin3,
                           const float* h_spacing3, const float* h_plane_origin3,
                           const float* h_plane_normal3, void* d_workspace,
                           size_t workspace_bytes, int64_t* h_tris, int64_t* h_points,
                           void* stream) {
  VolGeom g;
  FieldPlane pl;
  int rc = make_slice(nx, ny, nz, h_origin3, h_spacing3, h_plane_origin3, h_plane_normal3, g, pl);
  if (rc) return rc;
  Workspace L;
  if ((rc = check_ws(g, workspace_bytes, L, d_workspace))) return rc;
  if (!h_tris || !h_points) {
    set_error("dax_hip_mc_slice_count: h_tris and h_points are required");
    return DAX_HIP_BAD_VALUE;
  }
  hipStream_t s = (hipStream_t)stream;
  if ((rc = launch_bits_plane(g, pl, (char*)d_workspace, L, s))) return rc;
  return count_sync(g, (char*)d_workspace, L, tuning_for(nx, ny, nz), h_tris, h_points, s);
}

int dax_hip_mc_slice_generate(int64_t nx, int64_t ny, int64_t nz, const float* h_origin3,
                              const float* h_spacing3, const float* h_plane_origin3,
                              const float* h_plane_normal3, unsigned flags,
                              const void* d_workspace, size_t workspace_bytes, float* d_vertices,
                              float* d_normals, int32_t* d_conn, uint32_t* d_edges,
                              int32_t* d_interp_first, int32_t* d_interp_second,
                              float* d_interp_weight, int64_t cap_points, int64_t cap_tris,
                              int64_t* d_counts, void* stream) {
  VolGeom g;
  FieldPlane pl;
  int rc = make_slice(nx, ny, nz, h_origin3, h_spacing3, h_plane_origin3, h_plane_normal3, g, pl);
  if (rc) return rc;
  Workspace L;
  if ((rc = check_ws(g, workspace_bytes, L, (void*)d_workspace))) return rc;
  static const float kNoField = 0.0f;  // the slice reads no field
  if ((rc = check_outputs(g, &kNoField, flags, d_vertices, d_conn, d_edges, d_counts))) return rc;
  OutPtrs o{d_vertices, d_normals, d_conn, d_edges, d_interp_first, d_interp_second,
            d_interp_weight};
  return launch_generate_src(g, pl, (const char*)d_workspace, L, flags, o, cap_points, cap_tris,
                             d_counts, tuning_for(nx, ny, nz), (hipStream_t)stream);
}

int dax_hip_mc_slice(int64_t nx, int64_t ny, int64_t nz, const float* h_origin3,
                     const float* h_spacing3, const float* h_plane_origin3,
                     const float* h_plane_normal3, unsigned flags, void* d_workspace,
                     size_t workspace_bytes, float* d_vertices, float* d_normals, int32_t* d_conn,
                     uint32_t* d_edges, int32_t* d_interp_first, int32_t* d_interp_second,
                     float* d_interp_weight, int64_t cap_points, int64_t cap_tris,
                     int64_t* d_counts, void* stream) {
  VolGeom g;
  FieldPlane pl;
  int rc = make_slice(nx, ny, nz, h_origin3, h_spacing3, h_plane_origin3, h_plane_normal3, g, pl);
  if (rc) return rc;
  Workspace L;
  if ((rc = check_ws(g, workspace_bytes, L, d_workspace))) return rc;
  static const float kNoField = 0.0f;  // the slice reads no field
  if ((rc = check_outputs(g, &kNoField, flags, d_vertices, d_conn, d_edges, d_counts))) return rc;
  hipStream_t s = (hipStream_t)stream;
  char* ws = (char*)d_workspace;
  const Tuning tu = tuning_for(nx, ny, nz);
  OutPtrs o{d_vertices, d_normals, d_conn, d_edges, d_interp_first, d_interp_second,
            d_interp_weight};
  if ((rc = launch_bits_plane(g, pl, ws, L, s))) return rc;
  if ((rc = launch_scan(g, ws, L, tu, s))) return rc;
  return launch_generate_src(g, pl, ws, L, flags, o, cap_points, cap_tris, d_counts, tu, s);
}

int dax_hip_mc_read_counts(const int64_t* d_counts, int64_t cap_points, int64_t cap_tris,
                           int64_t* h_tris, int64_t* h_points, void* stream) {
  int64_t c[2];
  DAXHIP_CHECK(hipMemcpyAsync(c, d_counts, sizeof(c), hipMemcpyDeviceToHost, (hipStream_t)stream));
  DAXHIP_CHECK(hipStreamSynchronize((hipStream_t)stream));
  if (h_tris) *h_tris = c[0];
  if (h_points) *h_points = c[1];
  if (const int rc = check_totals(c[0], c[1])) return rc;
  if (c[0] > cap_tris || c[1] > cap_points) {
    set_error("dax_hip_mc: output needs %lld triangles / %lld points, capacity %lld / %lld",
              (long long)c[0], (long long)c[1], (long long)cap_tris, (long long)cap_points);
    return DAX_HIP_CAPACITY;
  }
  return DAX_HIP_OK;
}

int dax_hip_mc_cell_outputs(int64_t nx, int64_t ny, int64_t nz, const void* d_workspace,
                            size_t workspace_bytes, uint8_t* d_cases, int32_t* d_count,
                            int32_t* d_offsets, void* stream) {
  VolGeom g;
  int rc = make_geom(nx, ny, nz, nullptr, nullptr, 0.0f, g);
  if (rc) return rc;
  Workspace L;
  if ((rc = check_ws(g, workspace_bytes, L, (void*)d_workspace))) return rc;
  const char* ws = (const char*)d_workspace;
  const int64_t blocks = ceil_div(ceil_div(g.nwords, (int64_t)kCellWords) * 64, 256);
  if (blocks == 0) return DAX_HIP_OK;
  k_cell_outputs<<<dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream>>>(
      g, (const uint64_t*)(ws + L.off_bits), count_src(ws, L),
      (const Ctrl*)(ws + L.off_ctrl), d_cases, d_count, d_offsets);
  DAXHIP_LAUNCH_CHECK("k_cell_outputs");
  return DAX_HIP_OK;
}

int dax_hip_mc_interpolate_scalar(const float* d_in, const int32_t* d_first,
                                  const int32_t* d_second, const float* d_weight, int64_t n,
                                  float* d_out, void* stream) {
  if (n <= 0) return DAX_HIP_OK;
  k_interpolate_scalar<<<dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, (hipStream_t)stream>>>(
      d_in, d_first, d_second, d_weight, n, d_out);
  DAXHIP_LAUNCH_CHECK("k_interpolate_scalar");
  return DAX_HIP_OK;
}

int dax_hip_mc_interpolate_vec3(const float* d_in, const int32_t* d_first, const int32_t* d_second,
                                const float* d_weight, int64_t n, float* d_out, void* stream) {
  if (n <= 0) return DAX_HIP_OK;
  k_interpolate_vec3<<<dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, (hipStream_t)stream>>>(
      d_in, d_first, d_second, d_weight, n, d_out);
  DAXHIP_LAUNCH_CHECK("k_interpolate_vec3");
  return DAX_HIP_OK;
}

int dax_hip_point_gradient(const float* d_field, int64_t nx, int64_t ny, int64_t nz,
                           const float* h_spacing3, float* d_grad, void* stream) {
  VolGeom g;
  int rc = make_geom(nx, ny, nz, nullptr, h_spacing3, 0.0f, g);
  if (rc) return rc;
  if (!march_planes(nx * ny)) {
    const int64_t n = nx * ny * nz;
    k_point_gradient_flat<<<dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, (hipStream_t)stream>>>(
        g, n, d_field, d_grad);
    DAXHIP_LAUNCH_CHECK("k_point_gradient_flat");
    return DAX_HIP_OK;
  }
  const int64_t pb = ceil_div(nx * ny, (int64_t)256);
  const int planes = gradient_planes(pb, nz);
  k_point_gradient<<<dim3((unsigned)(pb * ceil_div(nz, (int64_t)planes))), dim3(256), 0,
                     (hipStream_t)stream>>>(g, planes, make_fast_div((uint32_t)pb), d_field,
                                            d_grad);
  DAXHIP_LAUNCH_CHECK("k_point_gradient");
  return DAX_HIP_OK;
}

int dax_hip_cell_gradient(const float* d_field, int64_t nx, int64_t ny, int64_t nz,
                          const float* h_origin3, const float* h_spacing3, float* d_grad,
                          void* stream) {
  VolGeom g;
  int rc = make_geom(nx, ny, nz, h_origin3, h_spacing3, 0.0f, g);
  if (rc) return rc;
  if (nx < 2 || ny < 2 || nz < 2) return DAX_HIP_OK;
  const FastDiv div_cx = make_fast_div((uint32_t)nx - 1u);
  if (!march_planes((nx - 1) * (ny - 1))) {
    const int64_t n = (nx - 1) * (ny - 1) * (nz - 1);
    k_cell_gradient_flat<<<dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, (hipStream_t)stream>>>(
        g, n, div_cx, make_fast_div((uint32_t)ny - 1u), d_field, d_grad);
    DAXHIP_LAUNCH_CHECK("k_cell_gradient_flat");
    return DAX_HIP_OK;
  }
  const int64_t pb = ceil_div((nx - 1) * (ny - 1), (int64_t)256);
  const int planes = gradient_planes(pb, nz - 1);
  k_cell_gradient<<<dim3((unsigned)(pb * ceil_div(nz - 1, (int64_t)planes))), dim3(256), 0,
                    (hipStream_t)stream>>>(g, planes, make_fast_div((uint32_t)pb), div_cx, d_field,
                                           d_grad);
  DAXHIP_LAUNCH_CHECK("k_cell_gradient");
  return DAX_HIP_OK;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Tuning and autotuning
namespace {

struct EventPair {
  hipEvent_t a = nullptr, b = nullptr;
  EventPair() {
    (void)hipEventCreate(&a);
    (void)hipEventCreate(&b);
  }
  ~EventPair() {
    if (a) (void)hipEventDestroy(a);
    if (b) (void)hipEventDestroy(b);
  }
  float ms() {
    float m = 0.0f;
    (void)hipEventSynchronize(b);
    (void)hipEventElapsedTime(&m, a, b);
    return m;
  }
};

}  // namespace

extern "C" {

int dax_hip_mc_set_tuning(int64_t nx, int64_t ny, int64_t nz, const int* h_params5) {
  if (!h_params5) {
    set_error("dax_hip_mc_set_tuning: NULL parameters");
    return DAX_HIP_BAD_VALUE;
  }
  Tuning t;
  t.cls_unroll = h_params5[0];
  t.cls_vec = h_params5[1];
  t.scan_sub = h_params5[2];
  t.gen_tile = h_params5[3];
  t.gen_xcd = h_params5[4];
  if (!valid_tuning(t)) {
    set_error("dax_hip_mc_set_tuning: invalid parameters {%d,%d,%d,%d,%d}", t.cls_unroll,
              t.cls_vec, t.scan_sub, t.gen_tile, t.gen_xcd);
    return DAX_HIP_BAD_VALUE;
  }
  std::lock_guard<std::mutex> lk(g_tune_mu);
  if (nx == 0 && ny == 0 && nz == 0) {
    g_tune_default = t;
    g_tune_default_set = true;
  } else {
    g_tune_cache[std::make_tuple(nx, ny, nz)] = t;
  }
  return DAX_HIP_OK;
}

int dax_hip_mc_get_tuning(int64_t nx, int64_t ny, int64_t nz, int* h_params5) {
  const Tuning t = (nx == 0 && ny == 0 && nz == 0) ? g_tune_default : tuning_for(nx, ny, nz);
  h_params5[0] = t.cls_unroll;
  h_params5[1] = t.cls_vec;
  h_params5[2] = t.scan_sub;
  h_params5[3] = t.gen_tile;
  h_params5[4] = t.gen_xcd;
  return DAX_HIP_OK;
}

int dax_hip_mc_tuning_save(const char* path) {
  FILE* fp = fopen(path, "w");
  if (!fp) {
    set_error("dax_hip_mc_tuning_save: cannot open %s", path);
    return DAX_HIP_BAD_VALUE;
  }
  std::lock_guard<std::mutex> lk(g_tune_mu);
  fprintf(fp, "# nx ny nz classify_unroll classify_vec scan_sub gen_tile gen_xcd\n");
  for (const auto& kv : g_tune_cache)
    fprintf(fp, "%lld %lld %lld %d %d %d %d %d\n", (long long)std::get<0>(kv.first),
            (long long)std::get<1>(kv.first), (long long)std::get<2>(kv.first), kv.second.cls_unroll,
            kv.second.cls_vec, kv.second.scan_sub, kv.second.gen_tile, kv.second.gen_xcd);
  fclose(fp);
  return DAX_HIP_OK;
}

int dax_hip_mc_tuning_load(const char* path) {
  FILE* fp = fopen(path, "r");
  if (!fp) {
    set_error("dax_hip_mc_tuning_load: cannot open %s", path);
    return DAX_HIP_BAD_VALUE;
  }
  char line[256];
  while (fgets(line, sizeof(line), fp)) {
    if (line[0] == '#') continue;
    long long x, y, z;
    Tuning t;
    if (sscanf(line, "%lld %lld %lld %d %d %d %d %d", &x, &y, &z, &t.cls_unroll, &t.cls_vec,
               &t.scan_sub, &t.gen_tile, &t.gen_xcd) == 8 &&
        valid_tuning(t)) {
      std::lock_guard<std::mutex> lk(g_tune_mu);
      g_tune_cache[std::make_tuple((int64_t)x, (int64_t)y, (int64_t)z)] = t;
    }
  }
  fclose(fp);
  return DAX_HIP_OK;
}

int dax_hip_mc_autotune(const float* d_field, int64_t nx, int64_t ny, int64_t nz, float iso,
                        unsigned flags, void* d_workspace, size_t workspace_bytes,
                        float* d_vertices, float* d_normals, int32_t* d_conn, uint32_t* d_edges,
                        int64_t cap_points, int64_t cap_tris, int64_t* d_counts, int reps,
                        int* h_best5, float* h_best_ms3, void* stream) {
  VolGeom g;
  int rc = make_geom(nx, ny, nz, nullptr, nullptr, iso, g);
  if (rc) return rc;
  Workspace L;
  if ((rc = check_ws(g, workspace_bytes, L, d_workspace))) return rc;
  if ((rc = check_outputs(g, d_field, flags, d_vertices, d_conn, d_edges, d_counts))) return rc;
  if (reps < 1) reps = 1;
  hipStream_t s = (hipStream_t)stream;
  char* ws = (char*)d_workspace;
  OutPtrs o{d_vertices, d_normals, d_conn, d_edges, nullptr, nullptr, nullptr};
  Tuning best = tuning_for(nx, ny, nz);
  EventPair ev;

  // classify variants (one for rows that are not whole words)
  std::vector<std::pair<int, int>> cls = {{best.cls_unroll, best.cls_vec}};
  if (nx % 64 == 0) cls = {{8, 1}, {16, 1}, {32, 1}, {2, 4}, {4, 4}, {8, 4}};
  float best_ms[3] = {1e30f, 1e30f, 1e30f};
  for (auto uv : cls) {
    Tuning t = best;
    t.cls_unroll = uv.first;
    t.cls_vec = uv.second;
    if ((rc = launch_bits(g, d_field, ws, L, t, s))) return rc;  // warm
    DAXHIP_CHECK(hipEventRecord(ev.a, s));
    for (int r = 0; r < reps; ++r)
      if ((rc = launch_bits(g, d_field, ws, L, t, s))) return rc;
    DAXHIP_CHECK(hipEventRecord(ev.b, s));
    const float ms = ev.ms() / reps;
    if (ms < best_ms[0]) {
      best_ms[0] = ms;
      best.cls_unroll = t.cls_unroll;
      best.cls_vec = t.cls_vec;
    }
  }
  // count/scan and generate variants together: the count block size decides
  // whether the count kernel classifies the generate tiles, and the tile
  // size the dispatch order the scan block builds (and its cost).  Each
  // repetition follows a classify, as in the forward; events split the
  // scan's time from generate's.
  EventPair ev2;
  const Tuning base = best;
  for (int sub : {1, 2, 4, 8}) {
    for (int tv = 0; tv < 10; ++tv) {
      Tuning t = base;
      t.scan_sub = sub;
      t.gen_tile = 64 << (tv % 5);
      t.gen_xcd = tv / 5;
      float ts = 0.0f, tg = 0.0f;
      for (int r = 0; r < reps; ++r) {
        if ((rc = launch_bits(g, d_field, ws, L, base, s))) return rc;
        DAXHIP_CHECK(hipEventRecord(ev.a, s));
        if ((rc = launch_scan(g, ws, L, t, s))) return rc;
        DAXHIP_CHECK(hipEventRecord(ev2.a, s));
        if ((rc = launch_generate(g, d_field, ws, L, flags, o, cap_points, cap_tris, d_counts, t,
                                  s)))
          return rc;
        DAXHIP_CHECK(hipEventRecord(ev.b, s));
        DAXHIP_CHECK(hipEventSynchronize(ev.b));
        float m1 = 0.0f, m2 = 0.0f;
        DAXHIP_CHECK(hipEventElapsedTime(&m1, ev.a, ev2.a));
        DAXHIP_CHECK(hipEventElapsedTime(&m2, ev2.a, ev.b));
        ts += m1;
        tg += m2;
      }
      ts /= reps;
      tg /= reps;
      if (ts + tg < best_ms[1] + best_ms[2]) {
        best_ms[1] = ts;
        best_ms[2] = tg;
        best.scan_sub = sub;
        best.gen_tile = t.gen_tile;
        best.gen_xcd = t.gen_xcd;
      }
    }
  }
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_tune_cache[std::make_tuple(nx, ny, nz)] = best;
  }
  if (h_best5) {
    h_best5[0] = best.cls_unroll;
    h_best5[1] = best.cls_vec;
    h_best5[2] = best.scan_sub;
    h_best5[3] = best.gen_tile;
    h_best5[4] = best.gen_xcd;
  }
  if (h_best_ms3)
    for (int i = 0; i < 3; ++i) h_best_ms3[i] = best_ms[i];
  return DAX_HIP_OK;
}

}  // extern "C"

