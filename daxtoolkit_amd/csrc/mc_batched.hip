// Batched marching cubes: many independent volumes (uneven extents,
// per-volume isovalue, origin and spacing) in one word space.  No reference
// counterpart (Dax runs one grid per dispatcher call).
//
// Layout: the volumes' fields are concatenated (volume v at field_off[v]);
// their row words are concatenated in volume order (word_off[v]).  Tiles of
// 256 row words never straddle a volume; a table maps tile -> (volume, first
// local word).  Every tile is counted as two count tiles, whose prefixes run
// over all tiles; subtracting the prefix of the volume's first tile makes the
// numbering per volume -- a segmented scan without segment flags.  Outputs
// are concatenated in volume order; connectivity is local to each volume;
// per-volume {first triangle, first point} offsets are written beside the
// counts.
//
// The four launches of a forward are graph-capturable (no host read-back).
#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include "mc_adjoint.h"
#include "mc_kernels.h"

namespace daxhip {
namespace mc {

struct TileRef {
  int32_t vol;
  int32_t w0;  // first row word, local to the volume
};

// The tile table is built at prepare.  The launch shapes over it are tuned.
constexpr int kBatchGenTile = 256;
// Threads per generate tile: one per word; a batch has tiles enough, so more
// waves per tile only stage the same words for fewer outputs each (256 volumes
// of 32..160 points an axis, forward + adjoint: 1077 us, 1133 with 512
// threads, 1250 with 1024).
constexpr int kBatchGenThreads = 256;

// Tiles of one launch: a launch takes fewer than 2^32 threads, and the tiles of
// more volumes than that go over several.
constexpr int64_t kLaunchTiles = 1 << 23;

// Launch shapes of the batch forward, picked by dax_hip_mc_batch_autotune
// and cached per batch shape class: classify unroll (row words per wave
// step, a float4 load in flight per thread for two of them) and persistent
// blocks per CU, threads per count block (a wave per tile), generate's
// XCD-contiguous tile order.  gen_blocks has no effect (generate runs a block
// per tile) and is kept, and checked, for callers that set it.
struct BatchTuning {
  int32_t cls_unroll, cls_blocks, scan_threads, gen_blocks, gen_xcd, pad;
};
constexpr BatchTuning kBatchTuningDefault{16, 4, 256, 4, 1, 0};
bool valid_batch_tuning(const BatchTuning& t) {
  return (t.cls_unroll == 8 || t.cls_unroll == 16 || t.cls_unroll == 32) &&
         (t.cls_blocks == 2 || t.cls_blocks == 4 || t.cls_blocks == 8) &&
         (t.scan_threads == 256 || t.scan_threads == 512 || t.scan_threads == 1024) &&
         (t.gen_blocks == 2 || t.gen_blocks == 4 || t.gen_blocks == 8) &&
         (t.gen_xcd == 0 || t.gen_xcd == 1);
}

struct BatchLayout {
  size_t off_vols, off_gen_tiles, off_bits, off_vol_first, off_lpre,
      off_tloc, off_bsum, off_bpre, off_ctrl, off_ends, off_end_pre, off_end_sum, off_end_tile,
      off_end_base, bytes;
  int64_t nvols, nwords, ngen;
};

BatchLayout batch_layout(int64_t nvols, const int64_t* dims) {
  BatchLayout L;
  L.nvols = nvols;
  L.nwords = 0;
  L.ngen = 0;
  for (int64_t v = 0; v < nvols; ++v) {
    const int64_t w = ceil_div(dims[3 * v], 64) * dims[3 * v + 1] * dims[3 * v + 2];
    L.nwords += w;
    L.ngen += ceil_div(w, kBatchGenTile);
  }
  size_t off = 0;
  L.off_vols = off;
  off = align_up(off + (size_t)nvols * sizeof(VolGeom), 256);
  L.off_gen_tiles = off;
  off = align_up(off + (size_t)L.ngen * sizeof(TileRef), 256);
  L.off_bits = off;
  off = align_up(off + (size_t)(L.nwords + 1) * 8, 256);
  L.off_vol_first = off;
  off = align_up(off + (size_t)nvols * 4, 256);
  L.off_lpre = off;
  off = align_up(off + (size_t)L.ngen * kBatchGenTile * 4, 256);
  // two count tiles per tile, and the entry after the last of a full block
  L.off_tloc = off;
  off = align_up(off + (size_t)(2 * L.ngen + 1) * 8, 256);
  L.off_bsum = off;
  off = align_up(off + (size_t)(L.ngen + 1) * 8, 256);
  L.off_bpre = off;
  off = align_up(off + (size_t)(L.ngen + 1) * 8, 256);
  L.off_ctrl = off;
  off = align_up(off + sizeof(Ctrl), 256);
  L.off_ends = off;  // the adjoint's endpoint words, their prefixes, the tiles' sums and prefixes
  off = align_up(off + (size_t)L.nwords * 8, 256);
  L.off_end_pre = off;
  off = align_up(off + (size_t)L.nwords * 2, 256);
  L.off_end_sum = off;
  off = align_up(off + (size_t)L.ngen * 4, 256);
  L.off_end_tile = off;
  off = align_up(off + (size_t)L.ngen * 4, 256);
  L.off_end_base = off;  // the count tiles' vertex bases
  off = align_up(off + (size_t)L.ngen * 8, 256);
  L.bytes = off;
  return L;
}

// Header at the start of the workspace: the layout, so launches need only
// the workspace pointer after prepare.
struct BatchHeader {
  int64_t magic, nvols, nwords, ngen, max_wpr;
  size_t off_vols, off_gen_tiles, off_bits, off_vol_first, off_lpre,
      off_tloc, off_bsum, off_bpre, off_ctrl, off_ends, off_end_pre, off_end_sum, off_end_tile,
      off_end_base, bytes;
  BatchTuning tune;
};
constexpr int64_t kBatchMagic = 0x4441584842415443LL;  // "DAXHBATC"
constexpr size_t kBatchHeaderBytes = 256;
static_assert(sizeof(BatchHeader) <= kBatchHeaderBytes, "header fits its reserved bytes");

template <int LOADS>
__global__ __launch_bounds__(256) void k_batch_classify(const VolGeom* __restrict__ vols,
                                                        const TileRef* __restrict__ tiles,
                                                        int64_t ntiles,
                                                        const float* __restrict__ fields,
                                                        uint64_t* __restrict__ bits) {
  __shared__ FlatLds<kBatchGenTile> sh;
  for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const TileRef tr = tiles[t];
    const VolGeom g = vols[tr.vol];
    const int64_t w_end = min((int64_t)tr.w0 + kBatchGenTile, g.nwords);
    classify_flat<kBatchGenTile, LOADS>(flat_rows(g), fields + g.field_off, bits + g.word_off,
                                        (uint32_t)tr.w0, (uint32_t)w_end, sh,
                                        [&](float v) { return v > g.iso; });
    __syncthreads();  // LDS reused by the next tile
  }
}

// Count: a wave per tile (two count tiles), WAVES tiles per block.  No block
// waits for another (a single pass with decoupled look-back over 1024-word
// tiles took 200 us for 256 volumes of 32..160 points an axis; this and the
// scan of the block sums take 34 + 6).
template <int WAVES>
__global__ __launch_bounds__(64 * WAVES) void k_batch_count(
    const VolGeom* __restrict__ vols, const TileRef* __restrict__ tiles, int64_t ntiles,
    const uint64_t* __restrict__ bits, uint32_t* __restrict__ lpre,
    unsigned long long* __restrict__ tloc, unsigned long long* __restrict__ bsum, int64_t blk0) {
  constexpr int kBlockTiles = 2 * WAVES;
  __shared__ unsigned long long s_ts[kBlockTiles];
  const int wv = threadIdx.x >> 6;
  const int64_t blk = blk0 + xcd_tile(blockIdx.x, gridDim.x);
  const int64_t t = blk * WAVES + wv;
  unsigned long long s0 = 0ull, s1 = 0ull;
  if (t < ntiles) {
    const TileRef tr = tiles[t];
    const VolGeom g = vols[tr.vol];
    const int64_t pair = tr.w0 / kBatchGenTile;
    count_tile_pair(g, bits + g.word_off, lpre + g.tile_off * kBatchGenTile, pair, 2 * pair + 2,
                    s0, s1);
  }
  if ((threadIdx.x & 63) == 0) {
    s_ts[2 * wv] = s0;
    s_ts[2 * wv + 1] = s1;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long run = 0ull;
    for (int i = 0; i < kBlockTiles; ++i) {
      const int64_t tile = blk * kBlockTiles + i;
      if (tile <= 2 * ntiles) tloc[tile] = run;
      run = add_vt(run, s_ts[i]);
    }
    bsum[blk] = run;
  }
}

__global__ __launch_bounds__(kTsumThreads) void k_batch_scan(
    const unsigned long long* __restrict__ bsum, unsigned long long* __restrict__ bpre, int64_t n,
    unsigned long long* __restrict__ tloc, int64_t n_ctiles, Ctrl* __restrict__ ctrl,
    int tpb_shift) {
  __shared__ uint32_t s_v[kTsumThreads / 64], s_t[kTsumThreads / 64];
  unsigned long long cv, ct;
  scan_block_sums(bsum, bpre, n, s_v, s_t, cv, ct);
  if (threadIdx.x == 0) {
    if ((n_ctiles & ((1 << tpb_shift) - 1)) == 0) tloc[n_ctiles] = 0ull;
    ctrl->total_v = cv;
    ctrl->total_t = ct;
    ctrl->tpb_shift = (uint32_t)tpb_shift;
  }
}

// The count kernel's prefixes of one volume.
__device__ __forceinline__ CountSrc volume_counts(const CountSrc& all, const VolGeom& g) {
  CountSrc cs = all;
  cs.lpre += g.tile_off * kBatchGenTile;
  cs.n_ctiles = 2 * ceil_div(g.nwords, (int64_t)kBatchGenTile);
  cs.ct0 = 2 * g.tile_off;
  return cs;
}

// Generate, a block per tile (persistent blocks looping over the tiles, four
// per CU: forward of 256 volumes 400 us, this 368).  The tile at a volume's
// start also writes the volume's {first triangle, first point} in the
// concatenated outputs and its first vertex for the adjoint.
template <bool dedup>
__global__ __launch_bounds__(kBatchGenThreads, 4) void k_batch_generate(
    const VolGeom* __restrict__ vols, const TileRef* __restrict__ tiles, int64_t ntiles,
    const float* __restrict__ fields, const uint64_t* __restrict__ bits, CountSrc all,
    const Ctrl* __restrict__ ctrl, OutPtrs out, unsigned flags, int64_t cap_points,
    int64_t cap_tris, int64_t* __restrict__ counts, int64_t* __restrict__ vol_offsets,
    uint32_t* __restrict__ vol_first, int xcd) {
  extern __shared__ uint64_t s_dyn[];
  const bool normals = (flags & DAX_HIP_MC_NORMALS) != 0 && out.normals != nullptr;
  const uint64_t total_v = ctrl->total_v, total_t = ctrl->total_t;
  const uint64_t n_points = dedup ? total_v : 3ull * total_t;
  if (blockIdx.x == 0 && threadIdx.x == 0 && counts) {
    counts[0] = (int64_t)total_t;
    counts[1] = (int64_t)n_points;
  }
  // too many ids for dax::Id or too little room: no output
  const bool emit = total_v <= 0x7fffffffull && 3ull * total_t <= 0x7fffffffull &&
                    (int64_t)total_t <= cap_tris && (int64_t)n_points <= cap_points;
  const TileRef tr = tiles[xcd ? xcd_tile_runs(blockIdx.x, ntiles) : (int64_t)blockIdx.x];
  const VolGeom g = vols[tr.vol];
  const CountSrc cs = volume_counts(all, g);
  const unsigned long long vol = ctile_prefix(cs, 0);
  const int64_t vbv = (int64_t)(uint32_t)vol, vbt = (int64_t)(vol >> 32);
  if (tr.w0 == 0 && threadIdx.x == 0) {
    vol_first[tr.vol] = (uint32_t)vbv;
    if (vol_offsets) {
      vol_offsets[2 * tr.vol + 0] = vbt;
      vol_offsets[2 * tr.vol + 1] = dedup ? vbv : 3 * vbt;
    }
  }
  if (!emit) return;
  generate_tile<kBatchGenTile, kBatchGenThreads, FieldArray, dedup>(
      g, FieldArray{fields + g.field_off}, bits + g.word_off, tr.w0, out, normals, vbv, vbt, s_dyn,
      cs, false);
}

// ---- batched adjoint --------------------------------------------------------
// The launches of the single volume's adjoint over generate's tile table.
__device__ __forceinline__ void batch_endpoint_words(
    const VolGeom* __restrict__ vols, const TileRef* __restrict__ tiles, int64_t ntiles,
    const uint64_t* __restrict__ bits, const CountSrc& all, const Ctrl* __restrict__ ctrl,
    const Endpoints& ep, const EdgeList& list, int64_t blk) {  // a wave per tile
  const int64_t t =
      blk * (kAdjThreads / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (edge_count(list) == 0 || t >= ntiles) return;  // wave-uniform
  const TileRef tr = tiles[t];
  const VolGeom g = vols[tr.vol];
  CountSrc cs = volume_counts(all, g);
  cs.tpb_shift = (int)ctrl->tpb_shift;
  endpoint_words_tile(g, bits + g.word_off, cs, ep, tr.w0);
}

__global__ __launch_bounds__(kAdjThreads) void k_batch_endpoint_words(
    const VolGeom* __restrict__ vols, const TileRef* __restrict__ tiles, int64_t ntiles,
    const uint64_t* __restrict__ bits, CountSrc all, const Ctrl* __restrict__ ctrl, Endpoints ep,
    EdgeList list) {
  batch_endpoint_words(vols, tiles, ntiles, bits, all, ctrl, ep, list, blockIdx.x);
}

// A thread per vertex; its volume by binary search over the volumes' first
// vertices, then the wave takes its volumes one at a time (one, as a rule),
// so that the geometry stays in scalar registers.  A block per tile of words
// instead leaves most lanes idle (73 vertices per tile in 256 volumes of
// 32..160 points an axis: 80 us; this: 58).  Blocks from vertex_blocks on form
// the endpoint words (WORDS).  Their registers leave the records six waves of
// eight, which costs many vertices more than a launch beside them saves: 1024
// volumes with 20 a word 8100 us against 59 + 7156, 256 volumes with one in
// three words 82 against 27 + 63.
constexpr int64_t kDenseWords = 4;  // vertices per row word from which they go apart
template <bool WORDS>
__global__ __launch_bounds__(256) void k_batch_records(
    const VolGeom* __restrict__ vols, int64_t nvols, const uint32_t* __restrict__ vol_first,
    const float* __restrict__ fields, const uint32_t* __restrict__ edges,
    const float* __restrict__ dldx, const float* __restrict__ dldn,
    EdgeList list, VertexAdj* __restrict__ out, const TileRef* __restrict__ tiles,
    int64_t ntiles, const uint64_t* __restrict__ bits, CountSrc all,
    const Ctrl* __restrict__ ctrl, Endpoints ep, int64_t vertex_blocks) {
  if (WORDS && (int64_t)blockIdx.x >= vertex_blocks)  // uniform
    return batch_endpoint_words(vols, tiles, ntiles, bits, all, ctrl, ep, list,
                                (int64_t)blockIdx.x - vertex_blocks);
  const int64_t U = edge_count(list);
  const int64_t u = xcd_tile(blockIdx.x, vertex_blocks) * blockDim.x + threadIdx.x;
  int64_t vol = -1;
  if (u < U) {  // the last volume whose first vertex is at most u
    int64_t lo = 0, hi = nvols;
    while (hi - lo > 1) {
      const int64_t mid = (lo + hi) >> 1;
      if ((int64_t)vol_first[mid] <= u)
        lo = mid;
      else
        hi = mid;
    }
    vol = lo;
  }
  uint64_t todo = __ballot(vol >= 0);
  while (todo) {
    const int v = __builtin_amdgcn_readlane((int)vol, __builtin_ctzll(todo));
    const bool mine = (int)vol == v;
    if (mine) vertex_adjoint(vols[v], fields, edges, dldx, dldn, u, out);
    todo &= ~__ballot(mine);
  }
}

static_assert(kAdjTile == kBatchGenTile, "the adjoint's tiles are the generate tiles");

template <int WW, bool FOLD>
__global__ __launch_bounds__(kAdjThreads) void k_batch_endpoint_sums(
    const VolGeom* __restrict__ vols, const TileRef* __restrict__ tiles,
    const uint64_t* __restrict__ bits, const uint32_t* __restrict__ lpre, Endpoints ep,
    const VertexAdj* __restrict__ adj, EdgeList list, f32x4* __restrict__ sums) {
  __shared__ uint8_t s_mark[kAdjThreads / 64][64];
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t blk = xcd_tile_runs(blockIdx.x, gridDim.x);
  const int64_t t = blk / kAdjTileBlocks<WW>, part = blk % kAdjTileBlocks<WW>;
  if (FOLD && blockIdx.x == 0 && threadIdx.x == 0) sums[0] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const uint32_t before = endpoints_before<FOLD>(ep, t, part == 0, list);
  const TileRef tr = tiles[t];
  const VolGeom g = vols[tr.vol];
  const int64_t ww = (int64_t)tr.w0 + part * kAdjBlockWords<WW> + wv * WW;
  if (ww < g.nwords)  // wave-uniform
    endpoint_sums_wave<WW>(g, bits + g.word_off, lpre + g.tile_off * kBatchGenTile, ep, adj, list,
                           sums, ww, before, s_mark[wv]);
}

template <int WW>
__global__ __launch_bounds__(kAdjThreads, kGatherWaves<WW>) void k_batch_point_gather(
    const VolGeom* __restrict__ vols, const TileRef* __restrict__ tiles,
    const uint64_t* __restrict__ bits, const uint32_t* __restrict__ lpre, Endpoints ep,
    const VertexAdj* __restrict__ adj, EdgeList list, const f32x4* __restrict__ sums,
    uint32_t last, float* __restrict__ dldf) {
  __shared__ GatherWave<WW> s_wave[kAdjThreads / 64];
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t blk = xcd_tile_runs(blockIdx.x, gridDim.x);
  const TileRef tr = tiles[blk / kAdjTileBlocks<WW>];
  const VolGeom g = vols[tr.vol];
  const int64_t ww =
      (int64_t)tr.w0 + blk % kAdjTileBlocks<WW> * kAdjBlockWords<WW> + wv * WW;
  if (ww < g.nwords)  // wave-uniform
    gather_wave<WW>(g, bits + g.word_off, lpre + g.tile_off * kBatchGenTile, ep, adj, list, sums,
                    last, dldf + g.field_off, ww, s_wave[wv]);
}

}  // namespace mc
}  // namespace daxhip

using namespace daxhip;
using namespace daxhip::mc;

namespace {

int persistent_blocks(int per_cu) {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus <= 0)
    cus = 256;
  return cus * per_cu;
}

// Tuning cache per batch shape class: (volumes, ceil(log2(row words)),
// widest row in words).
std::mutex g_btune_mu;
std::map<std::tuple<int64_t, int, int64_t>, BatchTuning> g_btune_cache;

std::tuple<int64_t, int, int64_t> batch_class(const BatchHeader& h) {
  int lg = 0;
  while ((1LL << lg) < h.nwords) ++lg;
  return std::make_tuple(h.nvols, lg, h.max_wpr);
}

// Device pointers of a prepared workspace.
struct BatchPtrs {
  const VolGeom* vols;
  const TileRef* gen_tiles;
  uint64_t* bits;
  uint32_t* vol_first;
  uint32_t* lpre;
  unsigned long long* tloc;
  unsigned long long* bsum;
  unsigned long long* bpre;
  Ctrl* ctrl;
};

BatchPtrs batch_ptrs(const BatchHeader& h, void* d_workspace) {
  char* body = (char*)d_workspace + kBatchHeaderBytes;
  return BatchPtrs{(const VolGeom*)(body + h.off_vols),
                   (const TileRef*)(body + h.off_gen_tiles),
                   (uint64_t*)(body + h.off_bits),
                   (uint32_t*)(body + h.off_vol_first),
                   (uint32_t*)(body + h.off_lpre),
                   (unsigned long long*)(body + h.off_tloc),
                   (unsigned long long*)(body + h.off_bsum),
                   (unsigned long long*)(body + h.off_bpre),
                   (Ctrl*)(body + h.off_ctrl)};
}

int batch_classify(const BatchHeader& h, const BatchPtrs& p, const float* d_fields,
                   const BatchTuning& t, hipStream_t s) {
  const dim3 grid((unsigned)persistent_blocks(t.cls_blocks)), blk(256);
  switch (t.cls_unroll) {
    case 8:
      k_batch_classify<4><<<grid, blk, 0, s>>>(p.vols, p.gen_tiles, h.ngen, d_fields, p.bits);
      break;
    case 32:
      k_batch_classify<16><<<grid, blk, 0, s>>>(p.vols, p.gen_tiles, h.ngen, d_fields, p.bits);
      break;
    default:
      k_batch_classify<8><<<grid, blk, 0, s>>>(p.vols, p.gen_tiles, h.ngen, d_fields, p.bits);
  }
  DAXHIP_LAUNCH_CHECK("k_batch_classify");
  return DAX_HIP_OK;
}

// log2 of the count tiles per count block.
int batch_count_shift(const BatchTuning& t) {
  return t.scan_threads == 1024 ? 5 : (t.scan_threads == 512 ? 4 : 3);
}

int batch_scan(const BatchHeader& h, const BatchPtrs& p, const BatchTuning& t, hipStream_t s) {
  const int waves = t.scan_threads / 64;
  const int64_t blocks = ceil_div(h.ngen, (int64_t)waves), most = kLaunchTiles / waves;
  const dim3 blk((unsigned)t.scan_threads);
  for (int64_t b0 = 0; b0 < blocks; b0 += most) {
    const dim3 grid((unsigned)std::min(most, blocks - b0));
    switch (waves) {
      case 8:
        k_batch_count<8><<<grid, blk, 0, s>>>(p.vols, p.gen_tiles, h.ngen, p.bits, p.lpre, p.tloc,
                                              p.bsum, b0);
        break;
      case 16:
        k_batch_count<16><<<grid, blk, 0, s>>>(p.vols, p.gen_tiles, h.ngen, p.bits, p.lpre, p.tloc,
                                               p.bsum, b0);
        break;
      default:
        k_batch_count<4><<<grid, blk, 0, s>>>(p.vols, p.gen_tiles, h.ngen, p.bits, p.lpre, p.tloc,
                                              p.bsum, b0);
    }
    DAXHIP_LAUNCH_CHECK("k_batch_count");
  }
  k_batch_scan<<<1, dim3(kTsumThreads), 0, s>>>(p.bsum, p.bpre, blocks, p.tloc, 2 * h.ngen, p.ctrl,
                                                batch_count_shift(t));
  DAXHIP_LAUNCH_CHECK("k_batch_scan");
  return DAX_HIP_OK;
}

int batch_generate(const BatchHeader& h, const BatchPtrs& p, const float* d_fields,
                   unsigned flags, const OutPtrs& o, int64_t cap_points, int64_t cap_tris,
                   int64_t* d_counts, int64_t* d_vol_offsets, const BatchTuning& t,
                   hipStream_t s) {
  const CountSrc cs{p.lpre, p.tloc, p.bpre, 0, 0, batch_count_shift(t)};
  const size_t lds = GenLayout<kBatchGenTile, kBatchGenThreads>((int)h.max_wpr).bytes();
  for (int64_t t0 = 0; t0 < h.ngen; t0 += kLaunchTiles) {
    const int64_t n = std::min(kLaunchTiles, h.ngen - t0);
    const dim3 grid((unsigned)n);
    if (flags & DAX_HIP_MC_DEDUP)
      k_batch_generate<true><<<grid, dim3(kBatchGenThreads), lds, s>>>(
          p.vols, p.gen_tiles + t0, n, d_fields, p.bits, cs, p.ctrl, o, flags, cap_points,
          cap_tris, d_counts, d_vol_offsets, p.vol_first, t.gen_xcd);
    else
      k_batch_generate<false><<<grid, dim3(kBatchGenThreads), lds, s>>>(
          p.vols, p.gen_tiles + t0, n, d_fields, p.bits, cs, p.ctrl, o, flags, cap_points,
          cap_tris, d_counts, d_vol_offsets, p.vol_first, t.gen_xcd);
    DAXHIP_LAUNCH_CHECK("k_batch_generate");
  }
  return DAX_HIP_OK;
}

// What the last two launches of a batch backward take.
struct BatchAdjoint {
  const VolGeom* vols;
  const TileRef* tiles;
  int64_t ntiles;
  const uint64_t* bits;
  const uint32_t* lpre;
  Endpoints ep;
  VertexAdj* adj;
  EdgeList list;
  f32x4* sums;
  float* dldf;
};

template <int WW>
int launch_batch_sums_gather(const BatchAdjoint& c, hipStream_t s) {
  const dim3 grid((unsigned)(c.ntiles * kAdjTileBlocks<WW>)), block(kAdjThreads);
  if (c.list.n_points > 0) {
    if (c.ntiles > kFoldTiles)
      k_batch_endpoint_sums<WW, false><<<grid, block, 0, s>>>(c.vols, c.tiles, c.bits, c.lpre, c.ep,
                                                              c.adj, c.list, c.sums);
    else
      k_batch_endpoint_sums<WW, true><<<grid, block, 0, s>>>(c.vols, c.tiles, c.bits, c.lpre, c.ep,
                                                             c.adj, c.list, c.sums);
    DAXHIP_LAUNCH_CHECK("k_batch_endpoint_sums");
  }
  k_batch_point_gather<WW><<<grid, block, 0, s>>>(c.vols, c.tiles, c.bits, c.lpre, c.ep, c.adj,
                                                  c.list, c.sums, last_slot(c.list.n_points),
                                                  c.dldf);
  DAXHIP_LAUNCH_CHECK("k_batch_point_gather");
  return DAX_HIP_OK;
}

}  // namespace

extern "C" {

size_t dax_hip_mc_batch_workspace_bytes(int64_t n_volumes, const int64_t* h_dims3) {
  if (n_volumes <= 0 || !h_dims3) return 0;
  return kBatchHeaderBytes + batch_layout(n_volumes, h_dims3).bytes;
}

// Writes the volume and tile tables into the workspace (synchronous upload).
int dax_hip_mc_batch_prepare(int64_t n_volumes, const int64_t* h_dims3,
                             const int64_t* h_field_offsets, const float* h_isos,
                             const float* h_origins3, const float* h_spacings3, void* d_workspace,
                             size_t workspace_bytes, void* h_header_out, void* stream) {
  if (n_volumes <= 0 || n_volumes > 0x7fffffffLL || !h_dims3 || !h_field_offsets || !h_isos) {
    set_error("dax_hip_mc_batch_prepare: bad volume description");
    return DAX_HIP_BAD_VALUE;
  }
  const BatchLayout L = batch_layout(n_volumes, h_dims3);
  if (!d_workspace || workspace_bytes < kBatchHeaderBytes + L.bytes) {
    set_error("dax_hip_mc_batch_prepare: workspace of %zu bytes, %zu needed", workspace_bytes,
              kBatchHeaderBytes + L.bytes);
    return DAX_HIP_BAD_VALUE;
  }
  std::vector<VolGeom> vols((size_t)n_volumes);
  std::vector<TileRef> gen_tiles;
  gen_tiles.reserve((size_t)L.ngen);
  int64_t word_off = 0;
  for (int64_t v = 0; v < n_volumes; ++v) {
    const int64_t nx = h_dims3[3 * v], ny = h_dims3[3 * v + 1], nz = h_dims3[3 * v + 2];
    if (nx < 1 || ny < 1 || nz < 1 || nx * ny * nz > (1LL << 30) || ceil_div(nx, 64) > kMaxWpr) {
      set_error("dax_hip_mc_batch_prepare: volume %lld has unsupported dims %lld x %lld x %lld",
                (long long)v, (long long)nx, (long long)ny, (long long)nz);
      return DAX_HIP_BAD_VALUE;
    }
    VolGeom& g = vols[(size_t)v];
    g.nx = (int32_t)nx;
    g.ny = (int32_t)ny;
    g.nz = (int32_t)nz;
    g.wpr = (int32_t)ceil_div(nx, 64);
    g.iso = h_isos[v];
    for (int d = 0; d < 3; ++d) {
      g.origin[d] = h_origins3 ? h_origins3[3 * v + d] : 0.0f;
      g.spacing[d] = h_spacings3 ? h_spacings3[3 * v + d] : 1.0f;
    }
    g.field_off = h_field_offsets[v];
    g.word_off = word_off;
    g.nwords = (int64_t)g.wpr * ny * nz;
    set_geom_divs(g);
    g.tile_off = (int64_t)gen_tiles.size();
    for (int64_t w = 0; w < g.nwords; w += kBatchGenTile) gen_tiles.push_back({(int32_t)v, (int32_t)w});
    word_off += g.nwords;
  }
  BatchHeader h;
  h.magic = kBatchMagic;
  h.nvols = n_volumes;
  h.nwords = L.nwords;
  h.ngen = L.ngen;
  h.max_wpr = 1;
  for (const VolGeom& g : vols) h.max_wpr = std::max<int64_t>(h.max_wpr, g.wpr);
  h.off_vols = L.off_vols;
  h.off_gen_tiles = L.off_gen_tiles;
  h.off_bits = L.off_bits;
  h.off_vol_first = L.off_vol_first;
  h.off_lpre = L.off_lpre;
  h.off_tloc = L.off_tloc;
  h.off_bsum = L.off_bsum;
  h.off_bpre = L.off_bpre;
  h.off_ends = L.off_ends;
  h.off_end_pre = L.off_end_pre;
  h.off_end_sum = L.off_end_sum;
  h.off_end_tile = L.off_end_tile;
  h.off_end_base = L.off_end_base;
  h.off_ctrl = L.off_ctrl;
  h.bytes = L.bytes;
  h.tune = kBatchTuningDefault;
  {
    std::lock_guard<std::mutex> lk(g_btune_mu);
    const auto it = g_btune_cache.find(batch_class(h));
    if (it != g_btune_cache.end()) h.tune = it->second;
  }
  hipStream_t s = (hipStream_t)stream;
  char* ws = (char*)d_workspace;
  char* body = ws + kBatchHeaderBytes;
  DAXHIP_CHECK(hipMemcpyAsync(ws, &h, sizeof(h), hipMemcpyHostToDevice, s));
  DAXHIP_CHECK(hipMemcpyAsync(body + L.off_vols, vols.data(), vols.size() * sizeof(VolGeom),
                              hipMemcpyHostToDevice, s));
  DAXHIP_CHECK(hipMemcpyAsync(body + L.off_gen_tiles, gen_tiles.data(),
                              gen_tiles.size() * sizeof(TileRef), hipMemcpyHostToDevice, s));
  DAXHIP_CHECK(hipStreamSynchronize(s));
  if (h_header_out) memcpy(h_header_out, &h, sizeof(h));
  return DAX_HIP_OK;
}

size_t dax_hip_mc_batch_header_bytes(void) { return sizeof(BatchHeader); }

// The batch forward: four launches, graph-capturable.  h_header is
// the header returned by prepare.  d_counts {T, U} totals; d_vol_offsets
// [n][2] {first triangle, first point} of each volume.
int dax_hip_mc_batch_forward(const float* d_fields, const void* h_header, void* d_workspace,
                             size_t workspace_bytes, unsigned flags, float* d_vertices,
                             float* d_normals, int32_t* d_conn, uint32_t* d_edges,
                             int64_t cap_points, int64_t cap_tris, int64_t* d_counts,
                             int64_t* d_vol_offsets, void* stream) {
  const BatchHeader* h = (const BatchHeader*)h_header;
  if (!h || h->magic != kBatchMagic || !d_workspace ||
      workspace_bytes < kBatchHeaderBytes + h->bytes) {
    set_error("dax_hip_mc_batch_forward: header/workspace not prepared");
    return DAX_HIP_BAD_VALUE;
  }
  if (!d_fields || !d_vertices || !d_conn || !d_counts) {
    set_error("dax_hip_mc_batch_forward: fields, vertices, connectivity and counts are required");
    return DAX_HIP_BAD_VALUE;
  }
  if (d_edges && !(flags & DAX_HIP_MC_DEDUP)) {
    set_error("dax_hip_mc_batch_forward: the compact edge list needs dedup");
    return DAX_HIP_BAD_VALUE;
  }
  hipStream_t s = (hipStream_t)stream;
  const BatchPtrs p = batch_ptrs(*h, d_workspace);
  const BatchTuning t = valid_batch_tuning(h->tune) ? h->tune : kBatchTuningDefault;
  int rc;
  if ((rc = batch_classify(*h, p, d_fields, t, s))) return rc;
  if ((rc = batch_scan(*h, p, t, s))) return rc;
  OutPtrs o{d_vertices, d_normals, d_conn, d_edges, nullptr, nullptr, nullptr};
  return batch_generate(*h, p, d_fields, flags, o, cap_points, cap_tris, d_counts, d_vol_offsets, t,
                        s);
}

// Launch shapes of a prepared batch: {classify unroll, classify blocks per
// CU, threads per count block, generate blocks per CU, generate XCD order}.
int dax_hip_mc_batch_set_tuning(void* h_header, const int* h_params5) {
  BatchHeader* h = (BatchHeader*)h_header;
  if (!h || h->magic != kBatchMagic || !h_params5) {
    set_error("dax_hip_mc_batch_set_tuning: header not prepared or NULL parameters");
    return DAX_HIP_BAD_VALUE;
  }
  const BatchTuning t{h_params5[0], h_params5[1], h_params5[2], h_params5[3], h_params5[4], 0};
  if (!valid_batch_tuning(t)) {
    set_error("dax_hip_mc_batch_set_tuning: invalid parameters {%d,%d,%d,%d,%d}", t.cls_unroll,
              t.cls_blocks, t.scan_threads, t.gen_blocks, t.gen_xcd);
    return DAX_HIP_BAD_VALUE;
  }
  h->tune = t;
  return DAX_HIP_OK;
}

int dax_hip_mc_batch_get_tuning(const void* h_header, int* h_params5) {
  const BatchHeader* h = (const BatchHeader*)h_header;
  if (!h || h->magic != kBatchMagic || !h_params5) {
    set_error("dax_hip_mc_batch_get_tuning: header not prepared or NULL parameters");
    return DAX_HIP_BAD_VALUE;
  }
  const BatchTuning t = valid_batch_tuning(h->tune) ? h->tune : kBatchTuningDefault;
  h_params5[0] = t.cls_unroll;
  h_params5[1] = t.cls_blocks;
  h_params5[2] = t.scan_threads;
  h_params5[3] = t.gen_blocks;
  h_params5[4] = t.gen_xcd;
  return DAX_HIP_OK;
}

// Times every launch shape of each phase on this batch (reps launches each,
// HIP events on `stream`; synchronous), keeps the fastest in the header and
// in the cache for the batch's shape class (later prepares of that class
// start from it).  h_best5: the choice; h_best_ms3: its phase times.
int dax_hip_mc_batch_autotune(const float* d_fields, void* h_header, void* d_workspace,
                              size_t workspace_bytes, unsigned flags, float* d_vertices,
                              float* d_normals, int32_t* d_conn, uint32_t* d_edges,
                              int64_t cap_points, int64_t cap_tris, int64_t* d_counts, int reps,
                              int* h_best5, float* h_best_ms3, void* stream) {
  BatchHeader* h = (BatchHeader*)h_header;
  if (!h || h->magic != kBatchMagic || !d_workspace ||
      workspace_bytes < kBatchHeaderBytes + h->bytes || !d_fields || !d_vertices || !d_conn ||
      !d_counts) {
    set_error("dax_hip_mc_batch_autotune: header/workspace not prepared or outputs missing");
    return DAX_HIP_BAD_VALUE;
  }
  if (reps < 1) reps = 1;
  hipStream_t s = (hipStream_t)stream;
  const BatchPtrs p = batch_ptrs(*h, d_workspace);
  OutPtrs o{d_vertices, d_normals, d_conn, d_edges, nullptr, nullptr, nullptr};
  BatchTuning best = valid_batch_tuning(h->tune) ? h->tune : kBatchTuningDefault;
  float best_ms[3] = {1e30f, 1e30f, 1e30f};
  hipEvent_t e0 = nullptr, e1 = nullptr;
  DAXHIP_CHECK(hipEventCreate(&e0));
  DAXHIP_CHECK(hipEventCreate(&e1));
  int rc = DAX_HIP_OK;
  auto elapsed = [&]() -> float {
    float m = 0.0f;
    (void)hipEventSynchronize(e1);
    (void)hipEventElapsedTime(&m, e0, e1);
    return m;
  };
  // classify
  for (int u : {8, 16, 32})
    for (int bpc : {2, 4, 8}) {
      BatchTuning t = best;
      t.cls_unroll = u;
      t.cls_blocks = bpc;
      if ((rc = batch_classify(*h, p, d_fields, t, s))) goto done;  // warm
      (void)hipEventRecord(e0, s);
      for (int r = 0; r < reps; ++r)
        if ((rc = batch_classify(*h, p, d_fields, t, s))) goto done;
      (void)hipEventRecord(e1, s);
      const float ms = elapsed() / reps;
      if (ms < best_ms[0]) {
        best_ms[0] = ms;
        best.cls_unroll = u;
        best.cls_blocks = bpc;
      }
    }
  // scan: each timed launch follows a classify, as in the forward
  for (int nt : {256, 512, 1024}) {
    BatchTuning t = best;
    t.scan_threads = nt;
    float total = 0.0f;
    for (int r = 0; r < reps; ++r) {
      if ((rc = batch_classify(*h, p, d_fields, best, s))) goto done;
      (void)hipEventRecord(e0, s);
      if ((rc = batch_scan(*h, p, t, s))) goto done;
      (void)hipEventRecord(e1, s);
      total += elapsed();
    }
    if (total / reps < best_ms[1]) {
      best_ms[1] = total / reps;
      best.scan_threads = nt;
    }
  }
  // generate over one classify + scan
  if ((rc = batch_classify(*h, p, d_fields, best, s))) goto done;
  if ((rc = batch_scan(*h, p, best, s))) goto done;
  for (int xcd : {0, 1}) {
      BatchTuning t = best;
      t.gen_xcd = xcd;
      if ((rc = batch_generate(*h, p, d_fields, flags, o, cap_points, cap_tris, d_counts, nullptr, t,
                               s)))
        goto done;
      (void)hipEventRecord(e0, s);
      for (int r = 0; r < reps; ++r)
        if ((rc = batch_generate(*h, p, d_fields, flags, o, cap_points, cap_tris, d_counts, nullptr, t,
                               s)))
          goto done;
      (void)hipEventRecord(e1, s);
      const float ms = elapsed() / reps;
      if (ms < best_ms[2]) {
        best_ms[2] = ms;
        best.gen_xcd = xcd;
      }
    }
  h->tune = best;
  {
    std::lock_guard<std::mutex> lk(g_btune_mu);
    g_btune_cache[batch_class(*h)] = best;
  }
  if (h_best5) {
    h_best5[0] = best.cls_unroll;
    h_best5[1] = best.cls_blocks;
    h_best5[2] = best.scan_threads;
    h_best5[3] = best.gen_blocks;
    h_best5[4] = best.gen_xcd;
  }
  if (h_best_ms3)
    for (int i = 0; i < 3; ++i) h_best_ms3[i] = best_ms[i];
done:
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return rc;
}

// Batched adjoint: dL/dfield of every volume (at the fields' offsets) from
// dL/dvertex and dL/dnormal of the concatenated outputs of the last batch
// forward on this workspace.  d_scratch: dax_hip_mc_backward_scratch_bytes
// (n_points).
int dax_hip_mc_batch_backward(const float* d_fields, const void* h_header,
                              const void* d_workspace, size_t workspace_bytes,
                              const uint32_t* d_edges, const int64_t* d_counts, int64_t n_points,
                              const float* d_dl_dvertices, const float* d_dl_dnormals,
                              void* d_scratch, size_t scratch_bytes, float* d_dl_dfields,
                              void* stream) {
  const BatchHeader* h = (const BatchHeader*)h_header;
  if (!h || h->magic != kBatchMagic || !d_workspace ||
      workspace_bytes < kBatchHeaderBytes + h->bytes) {
    set_error("dax_hip_mc_batch_backward: header/workspace not prepared");
    return DAX_HIP_BAD_VALUE;
  }
  if (h->ngen >= (1 << 24)) {
    set_error("dax_hip_mc_batch_backward: %lld tiles, fewer than 2^24 fit a launch",
              (long long)h->ngen);
    return DAX_HIP_BAD_VALUE;
  }
  if (h->max_wpr > kMaxGatherWpr) {
    set_error("dax_hip_mc_batch_backward: rows of %lld points exceed the %d the adjoint stages",
              (long long)h->max_wpr * 64, kMaxGatherWpr * 64);
    return DAX_HIP_BAD_VALUE;
  }
  const size_t need = n_points > 0 ? adjoint_scratch_bytes(n_points) : 0;
  if (n_points < 0 || scratch_bytes < need ||
      (n_points > 0 && (!d_scratch || !d_edges || !d_dl_dvertices || !d_dl_dnormals)) ||
      !d_fields || !d_dl_dfields) {
    set_error("dax_hip_mc_batch_backward: missing buffers or scratch smaller than %zu bytes",
              need);
    return DAX_HIP_BAD_VALUE;
  }
  hipStream_t s = (hipStream_t)stream;
  const char* body = (const char*)d_workspace + kBatchHeaderBytes;
  const VolGeom* vols = (const VolGeom*)(body + h->off_vols);
  const TileRef* gen_tiles = (const TileRef*)(body + h->off_gen_tiles);
  const uint64_t* bits = (const uint64_t*)(body + h->off_bits);
  const CountSrc cs{(const uint32_t*)(body + h->off_lpre),
                    (const unsigned long long*)(body + h->off_tloc),
                    (const unsigned long long*)(body + h->off_bpre), 0, 0, 0};
  // the endpoint words live in the workspace; every call on it writes the same
  // values there
  char* wb = const_cast<char*>(body);
  const Endpoints ep{(uint64_t*)(wb + h->off_ends), (uint16_t*)(wb + h->off_end_pre),
                     (uint32_t*)(wb + h->off_end_sum), (uint32_t*)(wb + h->off_end_tile),
                     (uint32_t*)(wb + h->off_end_base)};
  const BatchAdjoint call{vols, gen_tiles, h->ngen, bits, cs.lpre, ep,
                          (VertexAdj*)d_scratch,
                          EdgeList{d_counts, n_points},
                          (f32x4*)((char*)d_scratch + endpoint_sums_offset(n_points)),
                          d_dl_dfields};
  if (n_points > 0) {
    const int64_t vertex_blocks = ceil_div(n_points, (int64_t)kAdjThreads);
    const int64_t word_blocks = ceil_div(h->ngen, (int64_t)(kAdjThreads / 64));
    const uint32_t* vol_first = (const uint32_t*)(body + h->off_vol_first);
    const Ctrl* ctrl = (const Ctrl*)(body + h->off_ctrl);
    if (n_points > kDenseWords * h->nwords) {
      k_batch_endpoint_words<<<dim3((unsigned)word_blocks), kAdjThreads, 0, s>>>(
          vols, gen_tiles, h->ngen, bits, cs, ctrl, ep, call.list);
      DAXHIP_LAUNCH_CHECK("k_batch_endpoint_words");
      k_batch_records<false><<<dim3((unsigned)vertex_blocks), kAdjThreads, 0, s>>>(
          vols, h->nvols, vol_first, d_fields, d_edges, d_dl_dvertices, d_dl_dnormals, call.list,
          call.adj, gen_tiles, h->ngen, bits, cs, ctrl, ep, vertex_blocks);
    } else {
      k_batch_records<true><<<dim3((unsigned)(vertex_blocks + word_blocks)), kAdjThreads, 0, s>>>(
          vols, h->nvols, vol_first, d_fields, d_edges, d_dl_dvertices, d_dl_dnormals, call.list,
          call.adj, gen_tiles, h->ngen, bits, cs, ctrl, ep, vertex_blocks);
    }
    DAXHIP_LAUNCH_CHECK("k_batch_records");
    if (h->ngen > kFoldTiles)
      if (const int rc = launch_scan_endpoints(ep, h->ngen, call.list, call.sums, s)) return rc;
  }
  switch (adjoint_wave_words(h->nwords, h->ngen)) {
    case 8: return launch_batch_sums_gather<8>(call, s);
    case 32: return launch_batch_sums_gather<32>(call, s);
    default: return launch_batch_sums_gather<64>(call, s);
  }
}

// Capture of any sequence of this library's launches on `stream` (e.g. a
// batch forward followed by its backward) into one executable graph.
int dax_hip_graph_begin_capture(void* stream) {
  if (!stream) {
    set_error("dax_hip_graph_begin_capture: capture needs a non-null stream");
    return DAX_HIP_BAD_VALUE;
  }
  DAXHIP_CHECK(hipStreamBeginCapture((hipStream_t)stream, hipStreamCaptureModeThreadLocal));
  return DAX_HIP_OK;
}

int dax_hip_graph_end_capture(void* stream, void** h_graph_exec) {
  hipGraph_t graph = nullptr;
  DAXHIP_CHECK(hipStreamEndCapture((hipStream_t)stream, &graph));
  hipGraphExec_t exec = nullptr;
  const hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  if (e != hipSuccess) return check_hip(e, "hipGraphInstantiate");
  *h_graph_exec = exec;
  return DAX_HIP_OK;
}

// Baseline of the batched path: the same volumes, one single-volume forward
// (four launches) and, when upstream gradients are given, one single-volume
// backward (three launches, four on large volumes) per volume, written at the
// offsets of the batched outputs (h_vol_offsets, as the batched forward reports
// them).
int dax_hip_mc_volume_loop(int64_t n_volumes, const int64_t* h_dims3,
                           const int64_t* h_field_offsets, const float* h_isos,
                           const float* h_origins3, const float* h_spacings3,
                           const float* d_fields, unsigned flags, void* d_workspace,
                           size_t workspace_bytes, const int64_t* h_vol_offsets,
                           int64_t cap_points, int64_t cap_tris, float* d_vertices,
                           float* d_normals, int32_t* d_conn, uint32_t* d_edges,
                           int64_t* d_counts_scratch, const float* d_dl_dvertices,
                           const float* d_dl_dnormals, void* d_scratch, size_t scratch_bytes,
                           float* d_dl_dfields, void* stream) {
  if (n_volumes <= 0 || !h_dims3 || !h_field_offsets || !h_isos || !h_vol_offsets ||
      !d_counts_scratch) {
    set_error("dax_hip_mc_volume_loop: bad arguments");
    return DAX_HIP_BAD_VALUE;
  }
  const bool backward = d_dl_dfields != nullptr;
  for (int64_t v = 0; v < n_volumes; ++v) {
    const int64_t t0 = h_vol_offsets[2 * v], p0 = h_vol_offsets[2 * v + 1];
    const int64_t t1 = v + 1 < n_volumes ? h_vol_offsets[2 * v + 2] : cap_tris;
    const int64_t p1 = v + 1 < n_volumes ? h_vol_offsets[2 * v + 3] : cap_points;
    if (t0 < 0 || p0 < 0 || t1 < t0 || p1 < p0 || t1 > cap_tris || p1 > cap_points) {
      set_error("dax_hip_mc_volume_loop: volume %lld offsets outside the outputs", (long long)v);
      return DAX_HIP_BAD_VALUE;
    }
    const int64_t* d = h_dims3 + 3 * v;
    const float* o = h_origins3 ? h_origins3 + 3 * v : nullptr;
    const float* sp = h_spacings3 ? h_spacings3 + 3 * v : nullptr;
    const float* f = d_fields + h_field_offsets[v];
    int rc = dax_hip_mc_forward(f, d[0], d[1], d[2], o, sp, h_isos[v], flags, d_workspace,
                                workspace_bytes, d_vertices + 3 * p0,
                                d_normals ? d_normals + 3 * p0 : nullptr, d_conn + 3 * t0,
                                d_edges ? d_edges + p0 : nullptr, nullptr, nullptr, nullptr,
                                p1 - p0, t1 - t0, d_counts_scratch, stream);
    if (rc) return rc;
    if (backward) {
      rc = dax_hip_mc_backward(f, d[0], d[1], d[2], o, sp, h_isos[v], d_workspace,
                               workspace_bytes, d_edges ? d_edges + p0 : nullptr,
                               d_counts_scratch, p1 - p0,
                               d_dl_dvertices ? d_dl_dvertices + 3 * p0 : nullptr,
                               d_dl_dnormals ? d_dl_dnormals + 3 * p0 : nullptr,
                               d_scratch, scratch_bytes,
                               d_dl_dfields + h_field_offsets[v], stream);
      if (rc) return rc;
    }
  }
  return DAX_HIP_OK;
}

// ---- graphs: capture a launch sequence once, replay it -------------------
// Captures dax_hip_mc_batch_forward(args) on `stream` into an executable
// graph (h_graph_exec receives a hipGraphExec_t).
int dax_hip_mc_batch_graph_create(const float* d_fields, const void* h_header, void* d_workspace,
                                  size_t workspace_bytes, unsigned flags, float* d_vertices,
                                  float* d_normals, int32_t* d_conn, uint32_t* d_edges,
                                  int64_t cap_points, int64_t cap_tris, int64_t* d_counts,
                                  int64_t* d_vol_offsets, void* stream, void** h_graph_exec) {
  hipStream_t s = (hipStream_t)stream;
  if (!s) {
    set_error("dax_hip_mc_batch_graph_create: capture needs a non-null stream");
    return DAX_HIP_BAD_VALUE;
  }
  DAXHIP_CHECK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
  int rc = dax_hip_mc_batch_forward(d_fields, h_header, d_workspace, workspace_bytes, flags,
                                    d_vertices, d_normals, d_conn, d_edges, cap_points, cap_tris,
                                    d_counts, d_vol_offsets, stream);
  hipGraph_t graph = nullptr;
  hipError_t e = hipStreamEndCapture(s, &graph);
  if (rc) {
    if (graph) (void)hipGraphDestroy(graph);
    return rc;
  }
  if (e != hipSuccess) return check_hip(e, "hipStreamEndCapture");
  hipGraphExec_t exec = nullptr;
  e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  if (e != hipSuccess) return check_hip(e, "hipGraphInstantiate");
  *h_graph_exec = exec;
  return DAX_HIP_OK;
}

int dax_hip_graph_launch(void* graph_exec, void* stream) {
  DAXHIP_CHECK(hipGraphLaunch((hipGraphExec_t)graph_exec, (hipStream_t)stream));
  return DAX_HIP_OK;
}

int dax_hip_graph_destroy(void* graph_exec) {
  if (graph_exec) DAXHIP_CHECK(hipGraphExecDestroy((hipGraphExec_t)graph_exec));
  return DAX_HIP_OK;
}

}  // extern "C"
