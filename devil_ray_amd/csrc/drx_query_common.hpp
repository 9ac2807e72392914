// Helpers shared by the query (drx_query.hip) and integration (drx_integrate.hip) translation units.
#pragma once

#include "drx_common.hpp"
#include "drx_element.hpp"
#include "drx_wave.hpp"

namespace drx
{

// ---- arithmetic that must round like dray's float32 CPU path (no FMA contraction) --------------
__device__ __forceinline__ float ray_point (float o, float t, float d)
{
#pragma clang fp contract(off)
  return o + t * d;
}

__device__ __forceinline__ float mul_sub_nc (float a, float b, float c)
{
#pragma clang fp contract(off)
  return a * b - c;
}

__device__ __forceinline__ void blend_nc (float f[4], const float4 b)   // rendering/colors.hpp:15-23
{
#pragma clang fp contract(off)
  const float a = b.w * (1.f - f[3]);
  f[0] = f[0] + b.x * a;
  f[1] = f[1] + b.y * a;
  f[2] = f[2] + b.z * a;
  f[3] = a + f[3];
}

// DeviceColorMap::color for Float = double (device_color_map.hpp:61-77): clamp and normalise in double,
// the normalised value rounded to float32 before it is scaled to an index.
__device__ __forceinline__ int color_index64 (int size, double mn, double mx, double inv, double scalar)
{
#pragma clang fp contract(off)
  const double s = fmin (mx, fmax (mn, scalar));
  const double s2 = (scalar != scalar) ? mn : s;
  const float normalized = (float)((s2 - mn) * inv);
  int idx = (int)(normalized * (float)(size - 1));
  return min (max (idx, 0), size - 1);
}
__device__ __forceinline__ float4 color_lookup64 (const float4 *__restrict__ lut, int size, double mn, double mx,
                                                  double inv, double scalar)
{
  return lut[color_index64 (size, mn, mx, inv, scalar)];
}

// DeviceColorMap::color (device_color_map.hpp:61-77)
__device__ __forceinline__ int color_index (int size, float mn, float mx, float inv, float scalar)
{
#pragma clang fp contract(off)
  const float s = fminf (mx, fmaxf (mn, scalar));
  const float s2 = (scalar != scalar) ? mn : s;   // std::max(min, NaN) keeps min
  const float normalized = (s2 - mn) * inv;
  int idx = (int)(normalized * (float)(size - 1));
  return min (max (idx, 0), size - 1);
}
__device__ __forceinline__ float4 color_lookup (const float4 *__restrict__ lut, int size, float mn, float mx, float inv,
                                                float scalar)
{
  return lut[color_index (size, mn, mx, inv, scalar)];
}

static inline unsigned nblk (int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

#ifndef DRX_WAVES_PER_EU
#define DRX_WAVES_PER_EU 0   // 0: per-kernel choice below; otherwise a fixed minimum waves per SIMD
#endif

// Minimum waves per SIMD for the locate / integrate kernels (sets the VGPR budget: 5 -> 96, 4 -> 128).
// Measured on MI355X: order <= 3 walks run fastest at 5 (1024^2 render of a 64^3 order-3 mesh, 512
// samples per ray: 19.97 ms vs 22.37 ms at 4, some spills included; with FP64 polish, whose correction is
// an out-of-line call, 14.36 ms vs 16.40 ms at 4); order 4 and the learned start need the 128-register
// budget (2048^2 render of a 128^3 order-4 mesh, 1000 samples per ray: 297.5 ms at 4 vs 323 ms at 5).
#ifndef DRX_LEARNED_WAVES
#define DRX_LEARNED_WAVES 4   // learned-start integrate kernels (mode 3); 3 (no spills) measured slower
#endif
__host__ __device__ constexpr int waves_per_simd (int P, bool polish, int mode)
{
  return DRX_WAVES_PER_EU > 0 ? DRX_WAVES_PER_EU
                              : (mode == 3 ? DRX_LEARNED_WAVES : ((P >= 1 && P <= 3) ? 5 : 4));
}

// Compute units of device `dev` (cached per device; 256 if the query fails).
inline int compute_units (int dev)
{
  static int cus[16];
  if (dev < 0 || dev >= 16) return 256;
  if (!cus[dev])
  {
    int v = 0;
    cus[dev] = (hipDeviceGetAttribute (&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0) ? v : 256;
  }
  return cus[dev];
}

// Streamed batched-locate kernels (k_locate_stream, k_locate_mlp_stream): the integrate kernels' choice
// unless DRX_LOCATE_WAVES fixes it.
#ifndef DRX_LOCATE_WAVES
#define DRX_LOCATE_WAVES 0
#endif
__host__ __device__ constexpr int locate_waves_per_simd (int P, bool polish, int mode)
{
  return DRX_LOCATE_WAVES > 0 ? DRX_LOCATE_WAVES : (mode == 3 ? 4 : waves_per_simd (P, polish, mode));
}

static __global__ void k_fill_i32q (int32_t *p, int64_t n, int32_t v)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Order-preserving compaction in two passes over the items (keep (i): whether item i stays; put (i, k): writes it as
// the k-th kept one): kept items per block, then their places.  A block takes kCompactBlock items, each wavefront a
// quarter of them in a row.  One flag and one scan entry per item took two launches more and, for the 1.3 M partial
// slots of a 512^2 frame, 16 MB of traffic.  Up to kCompactSelfScan blocks (4 M items) each block of the second pass
// adds up the counts before its own, 16 loads per thread at most, which costs less than the launch of a scan (5 us and
// the gap); with more the counts are scanned first.
constexpr int kCompactThreads = 256, kCompactRounds = 4, kCompactBlock = kCompactThreads * kCompactRounds;
constexpr int kCompactSelfScan = 4096;
inline int32_t compact_blocks (int64_t n) { return (int32_t)((n + kCompactBlock - 1) / kCompactBlock); }

template <typename Keep> __device__ __forceinline__ void compact_count (int64_t n, int32_t *counts, Keep &&keep)
{
  __shared__ int32_t wcnt[kCompactThreads / 64];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t i0 = (int64_t)blockIdx.x * kCompactBlock + w * (64 * kCompactRounds) + lane;
  int32_t c = 0;
#pragma unroll
  for (int r = 0; r < kCompactRounds; ++r) c += __popcll (__ballot (i0 + 64 * r < n && keep (i0 + 64 * r)));
  if (lane == 0) wcnt[w] = c;
  __syncthreads ();
  if (threadIdx.x == 0) counts[blockIdx.x] = (wcnt[0] + wcnt[1]) + (wcnt[2] + wcnt[3]);
}

template <typename Keep, typename Put>
__device__ __forceinline__ void compact_put (int64_t n, const int32_t *counts, bool scanned, int32_t *total, Keep &&keep,
                                             Put &&put)
{
  __shared__ int32_t wcnt[kCompactThreads / 64], wbefore[kCompactThreads / 64];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t i0 = (int64_t)blockIdx.x * kCompactBlock + w * (64 * kCompactRounds) + lane;
  uint64_t b[kCompactRounds];
  int32_t c = 0;
#pragma unroll
  for (int r = 0; r < kCompactRounds; ++r)
  {
    b[r] = __ballot (i0 + 64 * r < n && keep (i0 + 64 * r));
    c += __popcll (b[r]);
  }
  int32_t before = 0;
  if (!scanned)
    for (int q = threadIdx.x; q < (int)blockIdx.x; q += kCompactThreads) before += counts[q];
  before = wave_scan_incl_add (before);
  if (lane == 63)
  {
    wcnt[w] = c;
    wbefore[w] = before;
  }
  __syncthreads ();
  int32_t k = scanned ? counts[blockIdx.x] : (wbefore[0] + wbefore[1]) + (wbefore[2] + wbefore[3]);
  if (threadIdx.x == 0 && blockIdx.x == gridDim.x - 1) *total = k + (wcnt[0] + wcnt[1]) + (wcnt[2] + wcnt[3]);
  for (int q = 0; q < w; ++q) k += wcnt[q];
#pragma unroll
  for (int r = 0; r < kCompactRounds; ++r)
  {
    if ((b[r] >> lane) & 1ull) put (i0 + 64 * r, k + __popcll (b[r] & ((1ull << lane) - 1)));
    k += __popcll (b[r]);
  }
}

static inline int check_mesh (const drx_mesh *m, int ncomp, const char *what)
{
  if (!m || !(m->data || (ncomp == 1 && m->data64))) return fail (DRX_ERR_ARG, "%s: null mesh", what);
  if (m->ncomp != ncomp) return fail (DRX_ERR_ARG, "%s: expected ncomp %d, got %d", what, ncomp, m->ncomp);
  if (ncomp == 3 && m->data64) return fail (DRX_ERR_ARG, "%s: FP64 blocks are for scalar fields only", what);
  if ((m->elem_order == nullptr) != (m->elem_offset == nullptr))
    return fail (DRX_ERR_ARG, "%s: mixed-order meshes need elem_order and elem_offset", what);
  if (!m->elem_order)
  {
    if (m->order < 1 || m->order > DRX_MAX_ORDER)
      return fail (DRX_ERR_ARG, "%s: order %d outside 1..%d", what, m->order, DRX_MAX_ORDER);
    if (m->stride != drx_mesh_stride (m->order, ncomp))
      return fail (DRX_ERR_ARG, "%s: stride %d does not match order %d", what, m->stride, m->order);
  }
  return DRX_OK;
}

// Whether the entry members were set by a caller that knows them (they came after the others, and a struct that a caller
// fills member by member need not be clear).
static inline bool has_entry_cells (const drx_bvh *b) { return b->entry_cells && b->entry_mark == drx_bvh_entry_mark (b); }

static inline int check_bvh (const drx_bvh *b, const char *what)
{
  if (!b || !b->inner_nodes || !b->leaf_pack) return fail (DRX_ERR_ARG, "%s: bvh needs inner_nodes and leaf_pack", what);
  if (b->n_leaves < 2) return fail (DRX_ERR_ARG, "%s: bvh has %d leaves (dray pads to >= 2)", what, b->n_leaves);
  if (has_entry_cells (b))
    for (int d = 0; d < 3; ++d)
      if (b->entry_bits[d] < 0 || b->entry_bits[d] > 16 || b->entry_bits[0] + b->entry_bits[1] + b->entry_bits[2] > 30)
        return fail (DRX_ERR_ARG, "%s: bvh entry_bits", what);
  return DRX_OK;
}

static inline LocateCfg make_cfg (const drx_mesh *m, const drx_bvh *b, const drx_locate_opts *o)
{
  LocateCfg c;
  c.nodes = (const float4 *)b->inner_nodes;
  c.wide = (const float4 *)b->wide_nodes;
  c.leaves = (const float4 *)b->leaf_pack;
  c.qnodes = (const uint4 *)b->qnodes;
  c.leaf_boxes = (const float4 *)b->leaf_boxes;
  for (int d = 0; d < 3; ++d)
  {
    c.q_org[d] = b->qgrid[d];
    c.q_inv[d] = b->qgrid[3 + d];
  }
  if (c.qnodes && !c.leaf_boxes) c.qnodes = nullptr;
  c.entry = c.qnodes && has_entry_cells (b) ? (const uint4 *)b->entry_cells : nullptr;
  for (int d = 0; d < 3; ++d) c.entry_bits[d] = c.entry ? b->entry_bits[d] : 0;
  c.centre = o && (o->init_mode == DRX_INIT_SUBREF_CENTRE || (o->init_mode == DRX_INIT_MLP && o->mlp_fallback == 1));
  c.starts = c.centre ? nullptr : (const float4 *)b->leaf_starts;
  c.mesh = m->data;
  c.offsets = m->elem_offset;
  c.orders = m->elem_order;
  c.stride = m->stride;
  c.polish = o ? (o->fp64_polish != 0) : false;
  c.cond_threshold = o ? o->cond_threshold : 1e4f;
  c.polished_out = o ? o->polished : nullptr;
  c.guess = (o && o->init_mode == DRX_INIT_GUESS) ? (const Location *)o->guess : nullptr;
  c.record = o ? (Location *)o->record : nullptr;
  c.samples_per_ray = o ? o->samples_per_ray : 0;
  return c;
}

} // namespace drx
