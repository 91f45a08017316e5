// Adjoint of the marching-cubes forward (no reference counterpart): the
// single-volume launches and C-ABI.  The math and the per-vertex / per-point
// device code are in mc_adjoint.h.
#include "mc_adjoint.h"

namespace daxhip {
namespace mc {

// Blocks [0, vertex_blocks): a thread per vertex; the rest: the endpoint words
// of a tile per wave (in a launch of their own they took as long: 1024^3 110 +
// 337 us against 451).
__global__ __launch_bounds__(kAdjThreads) void k_adjoint_records(
    VolGeom g, const float* __restrict__ field, const uint32_t* __restrict__ edges,
    const float* __restrict__ dldx, const float* __restrict__ dldn, EdgeList list,
    VertexAdj* __restrict__ out, const uint64_t* __restrict__ bits, CountSrc cs,
    const Ctrl* __restrict__ ctrl, Endpoints ep, int64_t vertex_blocks) {
  const int64_t U = edge_count(list);
  if ((int64_t)blockIdx.x >= vertex_blocks) {  // uniform
    const int64_t w0 = (((int64_t)blockIdx.x - vertex_blocks) * (kAdjThreads / 64) +
                        __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * kAdjTile;
    if (U == 0 || w0 >= g.nwords) return;  // wave-uniform
    cs.tpb_shift = (int)ctrl->tpb_shift;
    endpoint_words_tile(g, bits, cs, ep, w0);
    return;
  }
  // XCD-contiguous vertex ranges: vertices are in edge order, so the field
  // lines of neighbouring stencils stay in one XCD's L2
  const int64_t u = xcd_tile(blockIdx.x, vertex_blocks) * blockDim.x + threadIdx.x;
  if (u >= U) return;
  vertex_adjoint(g, field, edges, dldx, dldn, u, out);
}

template <int WW, bool FOLD>
__global__ __launch_bounds__(kAdjThreads) void k_endpoint_sums(
    VolGeom g, const uint64_t* __restrict__ bits, const uint32_t* __restrict__ lpre,
    Endpoints ep, const VertexAdj* __restrict__ adj, EdgeList list, f32x4* __restrict__ sums) {
  __shared__ uint8_t s_mark[kAdjThreads / 64][64];
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t blk = xcd_tile_runs(blockIdx.x, gridDim.x);
  const int64_t ww = blk * kAdjBlockWords<WW> + wv * WW;
  if (FOLD && blockIdx.x == 0 && threadIdx.x == 0) sums[0] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const uint32_t before = endpoints_before<FOLD>(ep, blk / kAdjTileBlocks<WW>,
                                                 blk % kAdjTileBlocks<WW> == 0, list);
  if (ww < g.nwords)  // wave-uniform
    endpoint_sums_wave<WW>(g, bits, lpre, ep, adj, list, sums, ww, before, s_mark[wv]);
}

template <int WW>
__global__ __launch_bounds__(kAdjThreads, kGatherWaves<WW>) void k_point_gather(
    VolGeom g, const uint64_t* __restrict__ bits, const uint32_t* __restrict__ lpre, Endpoints ep,
    const VertexAdj* __restrict__ adj, EdgeList list, const f32x4* __restrict__ sums,
    uint32_t last, float* __restrict__ dldf) {
  __shared__ GatherWave<WW> s_wave[kAdjThreads / 64];
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t ww = xcd_tile_runs(blockIdx.x, gridDim.x) * kAdjBlockWords<WW> + wv * WW;
  if (ww < g.nwords)  // wave-uniform
    gather_wave<WW>(g, bits, lpre, ep, adj, list, sums, last, dldf, ww, s_wave[wv]);
}

}  // namespace mc
}  // namespace daxhip

using namespace daxhip;
using namespace daxhip::mc;

namespace {

// What the last two launches of a backward take besides the geometry.
struct AdjointCall {
  const uint64_t* bits;
  CountSrc cs;
  Endpoints ep;
  EdgeList list;
  VertexAdj* adj;
  f32x4* sums;
  float* dldf;
};

template <int WW>
int launch_sums_gather(const VolGeom& g, const AdjointCall& c, int64_t tiles, hipStream_t s) {
  const dim3 grid((unsigned)ceil_div(g.nwords, (int64_t)kAdjBlockWords<WW>)), block(kAdjThreads);
  if (c.list.n_points > 0) {
    if (tiles > kFoldTiles)
      k_endpoint_sums<WW, false><<<grid, block, 0, s>>>(g, c.bits, c.cs.lpre, c.ep, c.adj, c.list,
                                                        c.sums);
    else
      k_endpoint_sums<WW, true><<<grid, block, 0, s>>>(g, c.bits, c.cs.lpre, c.ep, c.adj, c.list,
                                                       c.sums);
    DAXHIP_LAUNCH_CHECK("k_endpoint_sums");
  }
  k_point_gather<WW><<<grid, block, 0, s>>>(g, c.bits, c.cs.lpre, c.ep, c.adj, c.list, c.sums,
                                            last_slot(c.list.n_points), c.dldf);
  DAXHIP_LAUNCH_CHECK("k_point_gather");
  return DAX_HIP_OK;
}

}  // namespace

extern "C" {

int dax_hip_mc_backward_set_span_threshold(int64_t tiles_per_cu) {
  if (tiles_per_cu < 0) {
    set_error("dax_hip_mc_backward_set_span_threshold: negative threshold %lld",
              (long long)tiles_per_cu);
    return DAX_HIP_BAD_VALUE;
  }
  return DAX_HIP_OK;  // the gather has no dense tiles to choose a pass for
}

size_t dax_hip_mc_backward_scratch_bytes(int64_t n_points) {
  return n_points > 0 ? adjoint_scratch_bytes(n_points) : 0;
}

int dax_hip_mc_backward(const float* d_field, int64_t nx, int64_t ny, int64_t nz,
                        const float* h_origin3, const float* h_spacing3, float iso,
                        void* d_workspace, size_t workspace_bytes, const uint32_t* d_edges,
                        const int64_t* d_counts, int64_t n_points, const float* d_dl_dvertices,
                        const float* d_dl_dnormals, void* d_scratch, size_t scratch_bytes,
                        float* d_dl_dfield, void* stream) {
  if (nx < 1 || ny < 1 || nz < 1 || nx * ny * nz > (1LL << 30) ||
      (nx + 63) / 64 > kMaxGatherWpr) {
    set_error("dax_hip_mc_backward: unsupported grid %lld x %lld x %lld", (long long)nx,
              (long long)ny, (long long)nz);
    return DAX_HIP_BAD_VALUE;
  }
  VolGeom g;
  g.nx = (int32_t)nx;
  g.ny = (int32_t)ny;
  g.nz = (int32_t)nz;
  g.wpr = (int32_t)ceil_div(nx, 64);
  g.iso = iso;
  for (int d = 0; d < 3; ++d) {
    g.origin[d] = h_origin3 ? h_origin3[d] : 0.0f;
    g.spacing[d] = h_spacing3 ? h_spacing3[d] : 1.0f;
  }
  g.field_off = 0;
  g.word_off = 0;
  g.nwords = (int64_t)g.wpr * ny * nz;
  g.tile_off = 0;
  set_geom_divs(g);
  const Workspace L = workspace_layout(g.nwords);
  if (!d_workspace || workspace_bytes < L.bytes) {
    set_error("dax_hip_mc_backward: workspace of %zu bytes, %zu needed", workspace_bytes, L.bytes);
    return DAX_HIP_BAD_VALUE;
  }
  if (n_points < 0 || scratch_bytes < dax_hip_mc_backward_scratch_bytes(n_points) ||
      (n_points > 0 && (!d_scratch || !d_edges || !d_dl_dvertices || !d_dl_dnormals)) ||
      !d_field || !d_dl_dfield) {
    set_error("dax_hip_mc_backward: missing buffers or scratch smaller than %zu bytes",
              dax_hip_mc_backward_scratch_bytes(n_points));
    return DAX_HIP_BAD_VALUE;
  }
  hipStream_t s = (hipStream_t)stream;
  char* ws = (char*)d_workspace;
  const uint64_t* bits = (const uint64_t*)(ws + L.off_bits);
  const CountSrc cs{(const uint32_t*)(ws + L.off_counts),
                    (const unsigned long long*)(ws + L.off_tsum),
                    (const unsigned long long*)(ws + L.off_tpre), L.n_ctiles, 0, 0};
  // the endpoint words live in the workspace; every call on it writes the same
  // values there
  const Endpoints ep{(uint64_t*)(ws + L.off_ends), (uint16_t*)(ws + L.off_end_pre),
                     (uint32_t*)(ws + L.off_end_sum), (uint32_t*)(ws + L.off_end_tile),
                     (uint32_t*)(ws + L.off_end_base)};
  const AdjointCall call{bits, cs, ep, EdgeList{d_counts, n_points}, (VertexAdj*)d_scratch,
                         (f32x4*)((char*)d_scratch + endpoint_sums_offset(n_points)), d_dl_dfield};
  const int64_t tiles = ceil_div(g.nwords, (int64_t)kAdjTile);
  if (n_points > 0) {
    const int64_t vertex_blocks = ceil_div(n_points, (int64_t)kAdjThreads);
    const int64_t word_blocks = ceil_div(tiles, (int64_t)(kAdjThreads / 64));
    k_adjoint_records<<<dim3((unsigned)(vertex_blocks + word_blocks)), kAdjThreads, 0, s>>>(
        g, d_field, d_edges, d_dl_dvertices, d_dl_dnormals, call.list, call.adj, bits, cs,
        (const Ctrl*)(ws + L.off_ctrl), ep, vertex_blocks);
    DAXHIP_LAUNCH_CHECK("k_adjoint_records");
    if (tiles > kFoldTiles)
      if (const int rc = launch_scan_endpoints(ep, tiles, call.list, call.sums, s)) return rc;
  }
  switch (adjoint_wave_words(g.nwords, tiles)) {
    case 8: return launch_sums_gather<8>(g, call, tiles, s);
    case 32: return launch_sums_gather<32>(g, call, tiles, s);
    default: return launch_sums_gather<64>(g, call, tiles, s);
  }
}

}  // extern "C"
