// LBVH build for gfx950: per-element de Casteljau split into 33 sub-boxes, Morton codes, stable LSD
// radix sort, Karras tree, bottom-up refit, dray-layout emit.
//
// This file is compiled with -ffp-contract=off: every float operation here rounds exactly like dray's
// float32 CPU path, so the boxes, codes and the emitted tree are bit-identical to the reference's.
#include "drx_common.hpp"
#include "drx_wave.hpp"

#include <algorithm>
#include <cmath>
#include <vector>

namespace drx
{

// =============================================================================================
// Split: the 33 sub-boxes of every element.
// Semantics of construct_bvh (data_model/mesh_utils.cpp:557-670): 32 times pick the box of largest
// volume (surface area when the volume is 0; ties -> lowest index), split its SubRef at 0.5 along the
// longest reference axis (ties -> lowest axis, :482-506), de Casteljau-split the net (mother keeps the
// lower half, the copy at index `count` keeps the upper half; elem_ops.hpp:1346-1406), re-hull both.
// Then scale every box by 1.000001f about its centre (range.hpp:161-173).
//
// One workgroup per element.  A sub-box's net depends on its path from the element alone (the halves taken, along
// axis depth % 3: every split halves the longest reference axis, lowest first), so the boxes of the first five
// levels are split level by level, all boxes of a level in parallel, before it is known which of them the
// largest-first rule splits; the rule then runs on the 62 measures in registers.  A box below the fifth level that
// it picks (at least one: the 32nd split) is split on demand from its level-4 ancestor's net.  Nets and hulls are
// the ones the rule's own order gives, by the same operations.
//
// The rule's order (32 dependent splits of one net each, an argmax and LDS round trips per split) left a
// wavefront waiting on latency, and 33 nets of LDS per element few wavefronts per CU; only the 16 level-4 nets and
// one scratch net are held now (level 5 needs hulls only).  262,144 elements of order 3: 5.15 -> 1.08 ms (450 MB of
// output at copy rate: 0.1 ms); 110,592 of mixed orders 1-4: 5.37 -> 0.83 ms.  What is left is mostly the
// per-element rule and its on-demand splits, one wavefront each.
// =============================================================================================
constexpr int kSplitBoxes = 33;
constexpr int kSplitNets = 17;      // the level-4 nets and the scratch net of on-demand splits
constexpr int kSplitScratch = 16;
constexpr int kSplitExtras = 8;    // on-demand splits the ranked path holds

__device__ __forceinline__ float box_measure (const float *b)   // b: xmin,xmax,ymin,ymax,zmin,zmax
{
  const float l0 = b[1] - b[0], l1 = b[3] - b[2], l2 = b[5] - b[4];
  float v = 1.f;
  v *= l0;
  v *= l1;
  v *= l2;
  if (v == 0.f)
  {
    float a = 2.f * l0 * l1;
    a += 2.f * l1 * l2;
    a += 2.f * l2 * l0;
    v = a;
  }
  return v;
}

// Order-P layout: lanes per (net, component) group, one line per lane and pass, and the component stride of a
// net in LDS (a pad that staggers the groups' banks costs more occupancy than it saves: order 3, 4 floats: +9%).
template <int P> struct SplitOrd
{
  static constexpr int N1 = P + 1, LINES = N1 * N1, NPE = N1 * N1 * N1;
  static constexpr int G = P <= 3 ? 16 : P == 4 ? 32 : 64;
  static constexpr int CS = NPE;   // order 8: 17 nets just fit the LDS
};

// One line of a net: halves it along its axis (both halves in a[] and b[]).
template <int P> __device__ __forceinline__ void split_line (const float *m, int stride, float a[P + 1], float b[P + 1])
{
#pragma unroll
  for (int ii = 0; ii <= P; ++ii) a[ii] = b[ii] = m[ii * stride];
#pragma unroll
  for (int r = 1; r <= P; ++r)
  {
    // mother: new[ii] = .5 old[ii-1] + .5 old[ii] for ii >= r (descending, so old[ii-1] is still old)
#pragma unroll
    for (int ii = P; ii >= r; --ii) a[ii] = a[ii - 1] * (1.0f - 0.5f) + a[ii] * 0.5f;
    // daughter: new[ii] = .5 old[ii] + .5 old[ii+1] for ii <= P - r (ascending)
#pragma unroll
    for (int ii = 0; ii <= P - r; ++ii) b[ii] = b[ii] * (1.0f - 0.5f) + b[ii + 1] * 0.5f;
  }
}

// First dof and stride of line l along `axis` (the p+1 dofs along the axis, the other two indices fixed).
template <int P> __device__ __forceinline__ int line_base (int axis, int l)
{
  constexpr int N1 = P + 1;
  const int u = l % N1, v = l / N1;   // the two other indices, lowest axis first
  return axis == 0 ? N1 * l : axis == 1 ? u + N1 * N1 * v : l;
}
template <int P> __device__ __forceinline__ constexpr int line_stride (int axis)
{
  return axis == 0 ? 1 : axis == 1 ? P + 1 : (P + 1) * (P + 1);
}

// Min / max of the lanes' hull keys over a group of G lanes; the group's last lane ends with the result.  The
// lanes' hulls are never NaN (fminf / fmaxf from +-inf skip NaN values), so integer keys reduce them exactly.
template <int G> __device__ __forceinline__ float group_min (float f)
{
  int32_t v = row_reduce_min (float_key (f));
  if constexpr (G >= 32) v = min (v, dpp_move_i<0x142, 0xA> (v, v));
  if constexpr (G >= 64) v = min (v, dpp_move_i<0x143, 0xC> (v, v));
  return key_float (v);
}
template <int G> __device__ __forceinline__ float group_max (float f)
{
  int32_t v = row_reduce_max (float_key (f));
  if constexpr (G >= 32) v = max (v, dpp_move_i<0x142, 0xA> (v, v));
  if constexpr (G >= 64) v = max (v, dpp_move_i<0x143, 0xC> (v, v));
  return key_float (v);
}

// Splits component net `src` along `axis` with the lanes of one group (gl = lane in the group): the lower half to
// lo_dst, the upper to hi_dst (nullptr: not kept; lo_dst may be src), and the halves' hulls to lo_hull / hi_hull
// (min, max; nullptr: no hulls).  Lines are disjoint and each is read and written by one lane.
template <int P>
__device__ __forceinline__ void split_component (const float *src, float *lo_dst, float *hi_dst, int axis, int gl,
                                                 float *lo_hull, float *hi_hull)
{
  constexpr int G = SplitOrd<P>::G, LINES = SplitOrd<P>::LINES;
  const int stride = line_stride<P> (axis);
  float lo_a = INFINITY, hi_a = -INFINITY, lo_b = INFINITY, hi_b = -INFINITY;
#pragma unroll
  for (int l0 = 0; l0 < LINES; l0 += G)
  {
    const int l = l0 + gl;
    if (l < LINES)
    {
      const int base = line_base<P> (axis, l);
      float a[P + 1], b[P + 1];
      split_line<P> (src + base, stride, a, b);
#pragma unroll
      for (int ii = 0; ii <= P; ++ii)
      {
        if (lo_dst) lo_dst[base + ii * stride] = a[ii];
        if (hi_dst) hi_dst[base + ii * stride] = b[ii];
        lo_a = fminf (lo_a, a[ii]);
        hi_a = fmaxf (hi_a, a[ii]);
        lo_b = fminf (lo_b, b[ii]);
        hi_b = fmaxf (hi_b, b[ii]);
      }
    }
  }
  if (lo_hull)
  {
    lo_a = group_min<G> (lo_a);
    hi_a = group_max<G> (hi_a);
    lo_b = group_min<G> (lo_b);
    hi_b = group_max<G> (hi_b);
    if (gl == G - 1)
    {
      lo_hull[0] = lo_a;
      lo_hull[1] = hi_a;
      hi_hull[0] = lo_b;
      hi_hull[1] = hi_b;
    }
  }
}

// The speculative levels of one element: level D splits its 2^D boxes.  Box k of level D has its net in slot
// k * (16 >> D) and heap index 2^D + k; its lower child stays in the slot, its upper child takes the slot
// 16 >> (D + 1) above (level 4 keeps no nets).  hulls: 6 floats per heap index.
template <int P, int D>
__device__ __forceinline__ void split_level (float *nets, float *hulls, int group, int n_groups, int gl)
{
  constexpr int CS = SplitOrd<P>::CS, AXIS = D % 3, STEP = 16 >> D;
  for (int t = group; t < (3 << D); t += n_groups)
  {
    const int k = t / 3, c = t - 3 * k;
    float *net = nets + (k * STEP * 3 + c) * CS;
    float *h = hulls + 6 * (2 * ((1 << D) + k)) + 2 * c;
    if constexpr (D < 4)
      split_component<P> (net, net, net + (STEP / 2) * 3 * CS, AXIS, gl, h, h + 6);
    else
      split_component<P> (net, nullptr, nullptr, AXIS, gl, h, h + 6);
  }
}

__device__ __forceinline__ void split_wave_sync ()
{
  __builtin_amdgcn_fence (__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier ();
  __builtin_amdgcn_fence (__ATOMIC_ACQUIRE, "wavefront");
}

// On-demand split (one wavefront) of the box at `depth` >= 5 with path `path` (the halves taken, first split in
// the highest of the depth bits): its net is halved out of its level-4 ancestor's into the scratch net, then the
// hulls of its two halves go to hull_out[0..5] and [6..11].
template <int P>
__device__ __forceinline__ void split_deep (float *nets, float *hull_out, uint32_t path, int depth, int lane)
{
  constexpr int G = SplitOrd<P>::G, NG = 64 / G, CS = SplitOrd<P>::CS;
  const int group = lane / G, gl = lane % G;
  float *scratch = nets + kSplitScratch * 3 * CS;
  const float *src = nets + (path >> (depth - 4)) * 3 * CS;
  for (int d = 4; d < depth; ++d)
  {
    const bool upper = (path >> (depth - 1 - d)) & 1u;
    for (int c = group; c < 3; c += NG)
      split_component<P> (src + c * CS, upper ? nullptr : scratch + c * CS, upper ? scratch + c * CS : nullptr, d % 3, gl,
                          nullptr, nullptr);
    split_wave_sync ();
    src = scratch;
  }
  for (int c = group; c < 3; c += NG)
    split_component<P> (src + c * CS, nullptr, nullptr, depth % 3, gl, hull_out + 2 * c, hull_out + 6 + 2 * c);
  split_wave_sync ();
}

// Writes box k of the output: the hull scaled by 1.000001f about its centre, and the SubRef from the path (every
// split keeps one half along axis d % 3).
__device__ __forceinline__ void split_emit (int64_t k, const float *hull, uint32_t path, int depth,
                                            float *__restrict__ out_aabbs, float *__restrict__ out_subrefs)
{
  float ref[6] = { 0.f, 0.f, 0.f, 1.f, 1.f, 1.f };
  for (int d = 0; d < depth; ++d)
  {
    const bool upper = (path >> (depth - 1 - d)) & 1u;
    const int axis = d % 3;
#pragma unroll
    for (int q = 0; q < 3; ++q)
      if (q == axis)
      {
        const float split_pt = ref[q] * (1.0f - 0.5f) + ref[3 + q] * 0.5f;
        ref[q] = upper ? split_pt : ref[q];
        ref[3 + q] = upper ? ref[3 + q] : split_pt;
      }
  }
  const float s = (float)1.000001;
#pragma unroll
  for (int d = 0; d < 3; ++d)
  {
    float lo = hull[2 * d], hi = hull[2 * d + 1];
    if (!(lo > hi))
    {
      const float c = 0.5f * (lo + hi);
      const float delta = s * 0.5f * (hi - lo);
      const float v0 = c - delta, v1 = c + delta;
      lo = fminf (lo, v0);
      hi = fmaxf (hi, v0);
      lo = fminf (lo, v1);
      hi = fmaxf (hi, v1);
    }
    out_aabbs[6 * k + 2 * d] = lo;
    out_aabbs[6 * k + 2 * d + 1] = hi;
    out_subrefs[6 * k + d] = ref[d];
    out_subrefs[6 * k + 3 + d] = ref[3 + d];
  }
}

// The largest-first rule by ranks (one wavefront).  Where every box's measure is below its parent's and no two
// measures tie, the rule splits the 32 boxes of largest measure, in order of measure, so a box's rank among the 63
// is its place in that order: 63 broadcasts and compares instead of 32 dependent argmax reductions (262,144
// elements of order 3: 1.59 -> 1.08 ms).
// Box indices follow from the ranks: a lower child keeps its parent's index, an upper child takes the parent's
// place + 1.  Returns false, with nothing written, where that does not hold (ties, NaN measures, a
// box as large as its parent, a sixth-level box that would be split too, too many on-demand splits).
template <int P>
__device__ __forceinline__ bool split_ranked (float *nets, float *hulls, float *extra, float node_meas, int lane, int64_t k0,
                                              float *__restrict__ out_aabbs, float *__restrict__ out_subrefs)
{
  const int32_t key = lane <= 1 ? INT32_MAX : float_key (node_meas);
  if (__ballot (lane > 1 && !(node_meas == node_meas)) != 0) return false;
  int rank = 0;
#pragma unroll
  for (int h = 1; h < 64; ++h) rank += (__builtin_amdgcn_readlane (key, h) > key) ? 1 : 0;
  const bool split = lane >= 1 && rank < kSplitBoxes - 1;
  const uint64_t split_mask = __ballot (split);
  if (__popcll (split_mask) != kSplitBoxes - 1) return false;
  // each place 0..31 taken once (a tie leaves the next place free), each split box after its parent
  int32_t places = split ? (int32_t)(1u << rank) : 0;
  places |= dpp_perm_i<0xB1> (places);
  places |= dpp_perm_i<0x4E> (places);
  places |= dpp_perm_i<0x141> (places);
  places |= dpp_perm_i<0x140> (places);
  places |= dpp_move_i<0x142, 0xA> (0, places);
  places |= dpp_move_i<0x143, 0xC> (0, places);
  if (__builtin_amdgcn_readlane (places, 63) != -1) return false;
  const int parent_rank = __shfl (rank, lane >> 1, 64);
  if (__ballot (split && lane > 1 && parent_rank >= rank) != 0) return false;
  // box index: up to the first ancestor-or-self that is an upper child
  int index = 0;
  {
    int h = lane;
    bool open = lane > 1;
#pragma unroll
    for (int d = 0; d < 5; ++d)
    {
      const int pr = __shfl (rank, h >> 1, 64);
      if (open && (h & 1))
      {
        index = pr + 1;
        open = false;
      }
      h >>= 1;
      if (h <= 1) open = false;
    }
  }
  // on-demand splits of fifth-level boxes: their children must stay below the smallest box that is split
  const uint64_t deep = split_mask >> 32;
  const int n_deep = __popcll (deep);
  if (n_deep > kSplitExtras) return false;
  const int32_t least = __builtin_amdgcn_readlane (key, __ffsll ((unsigned long long)__ballot (split && rank == kSplitBoxes - 2)) - 1);
  uint64_t todo = deep;
  for (int x = 0; x < n_deep; ++x)
  {
    const int q = __ffsll ((unsigned long long)todo) - 1;
    todo &= todo - 1;
    split_deep<P> (nets, extra + 12 * x, (uint32_t)q, 5, lane);
  }
  {
    float b[6];
    bool big = false;
    if (lane < 2 * n_deep)
    {
#pragma unroll
      for (int q = 0; q < 6; ++q) b[q] = extra[6 * lane + q];
      const float m = box_measure (b);
      big = !(m == m) || float_key (m) >= least;
    }
    if (__ballot (big) != 0) return false;
  }
  const bool parent_split = lane > 1 && ((split_mask >> (lane >> 1)) & 1ull) != 0;
  if (parent_split && !split)
  {
    const int depth = 31 - __clz (lane);
    split_emit (k0 + index, hulls + 6 * lane, (uint32_t)(lane - (1 << depth)), depth, out_aabbs, out_subrefs);
  }
  // the children of the boxes split on demand: lanes 2x, 2x + 1
  {
    uint64_t m = deep;
    for (int x = 0; x < (lane >> 1); ++x) m &= m - 1;
    const int h = lane < 2 * n_deep ? 32 + __ffsll ((unsigned long long)m) - 1 : 1;
    const int hi = __shfl (index, h, 64), hr = __shfl (rank, h, 64);
    if (lane < 2 * n_deep)
      split_emit (k0 + ((lane & 1) ? hr + 1 : hi), extra + 6 * lane, (uint32_t)(2 * (h - 32) + (lane & 1)), 6, out_aabbs,
                  out_subrefs);
  }
  return true;
}

// The largest-first rule as dray runs it (one wavefront).
template <int P>
__device__ __forceinline__ void split_sequential (float *nets, float *hulls, float node_meas, int lane, int64_t k0,
                                                  float *__restrict__ out_aabbs, float *__restrict__ out_subrefs)
{
  // lane b (< 33): box b's path, depth and measure; the hull of a box from an on-demand split, else in `hulls`
  uint32_t my_path = 0;
  int my_depth = 0;
  float my_meas = 0.f, my_box[6];   // box 0 is the element, split first whatever its measure
#pragma unroll
  for (int q = 0; q < 6; ++q) my_box[q] = 0.f;
  bool own_box = false;
  for (int count = 1; count <= kSplitBoxes - 1; ++count)
  {
    // pick the box: dray's scan keeps the first strictly larger measure (ties -> lowest index; a NaN
    // never compares larger, and a NaN first measure is never replaced)
    int max_id = 0;
    {
      const float m0 = __int_as_float (__builtin_amdgcn_readfirstlane (__float_as_int (my_meas)));
      if (m0 == m0)
      {
        // integer keys: NaN measures and lanes beyond count can never be the maximum (box 0's key is a
        // number here, so the maximum is at least that)
        const int32_t cand = (lane < count && my_meas == my_meas) ? float_key (my_meas) : INT32_MIN;
        const int32_t M = wave_reduce_max (cand);
        const uint64_t hit = __ballot (lane < count && cand == M);
        max_id = __ffsll ((unsigned long long)hit) - 1;
      }
    }
    const uint32_t path = (uint32_t)__builtin_amdgcn_readlane ((int)my_path, max_id);
    const int depth = __builtin_amdgcn_readlane (my_depth, max_id);
    const bool low = lane == max_id, high = lane == count;
    if (low || high)
    {
      my_path = 2 * path + (high ? 1u : 0u);
      my_depth = depth + 1;
    }
    if (depth < 5)
    {
      const int h = 2 * ((1 << depth) + (int)path);
      const float ma = __int_as_float (__builtin_amdgcn_readlane (__float_as_int (node_meas), h));
      const float mb = __int_as_float (__builtin_amdgcn_readlane (__float_as_int (node_meas), h + 1));
      my_meas = low ? ma : high ? mb : my_meas;
    }
    else
    {
      split_deep<P> (nets, hulls, path, depth, lane);   // heap indices 0 and 1 are free
      if (low || high)
      {
#pragma unroll
        for (int q = 0; q < 6; ++q) my_box[q] = hulls[(high ? 6 : 0) + q];
        my_meas = box_measure (my_box);
        own_box = true;
      }
      split_wave_sync ();
    }
  }

  if (lane < kSplitBoxes)
  {
    if (!own_box)
    {
      const int h = (1 << my_depth) + (int)my_path;
#pragma unroll
      for (int q = 0; q < 6; ++q) my_box[q] = hulls[6 * h + q];
    }
    split_emit (k0 + lane, my_box, my_path, my_depth, out_aabbs, out_subrefs);
  }
}

template <int P, int WAVES>
__device__ __forceinline__ void split_element (const int32_t *__restrict__ ctrl_idx, const float *__restrict__ values,
                                               int64_t off, int e, float *nets, float *hulls, float *extra,
                                               float *__restrict__ out_aabbs, int32_t *__restrict__ out_prims,
                                               float *__restrict__ out_subrefs)
{
  constexpr int G = SplitOrd<P>::G, CS = SplitOrd<P>::CS, NPE = SplitOrd<P>::NPE;
  const int lane = threadIdx.x & 63;
  for (int d = threadIdx.x; d < NPE; d += 64 * WAVES)
  {
    const int64_t g = (int64_t)ctrl_idx[off + d] * 3;
#pragma unroll
    for (int c = 0; c < 3; ++c) nets[c * CS + d] = values[g + c];
  }
  __syncthreads ();
  const int group = threadIdx.x / G, n_groups = 64 * WAVES / G, gl = threadIdx.x % G;
  split_level<P, 0> (nets, hulls, group, n_groups, gl);
  __syncthreads ();
  split_level<P, 1> (nets, hulls, group, n_groups, gl);
  __syncthreads ();
  split_level<P, 2> (nets, hulls, group, n_groups, gl);
  __syncthreads ();
  split_level<P, 3> (nets, hulls, group, n_groups, gl);
  __syncthreads ();
  split_level<P, 4> (nets, hulls, group, n_groups, gl);
  __syncthreads ();
  if (threadIdx.x >= 64) return;

  // lane h (1..63): key of the measure of the box with heap index h (the element, h 1, is split first whatever it is)
  float node_meas;
  {
    float b[6];
#pragma unroll
    for (int q = 0; q < 6; ++q) b[q] = hulls[6 * lane + q];
    node_meas = box_measure (b);
  }
  const int64_t k0 = (int64_t)e * kSplitBoxes;
  if (!split_ranked<P> (nets, hulls, extra, node_meas, lane, k0, out_aabbs, out_subrefs))
    split_sequential<P> (nets, hulls, node_meas, lane, k0, out_aabbs, out_subrefs);
  if (lane < kSplitBoxes) out_prims[k0 + lane] = e;
}

template <int PMAX, int WAVES>
__global__ void __launch_bounds__ (64 * WAVES) k_split (const int32_t *__restrict__ ctrl_idx, const float *__restrict__ values,
                                                        const int32_t *__restrict__ orders,
                                                        const int64_t *__restrict__ offsets, int n_el,
                                                        float *__restrict__ out_aabbs, int32_t *__restrict__ out_prims,
                                                        float *__restrict__ out_subrefs)
{
  __shared__ __attribute__ ((aligned (16))) float nets[kSplitNets * 3 * SplitOrd<PMAX>::CS];
  __shared__ float hulls[64 * 6], extra[2 * kSplitExtras * 6];
  const int e = blockIdx.x;
  if (e >= n_el) return;
  const int64_t off = offsets ? offsets[e] : (int64_t)e * SplitOrd<PMAX>::NPE;
#define DRX_SPLIT_ELEMENT(P) split_element<P, WAVES> (ctrl_idx, values, off, e, nets, hulls, extra, out_aabbs, out_prims, out_subrefs)
  if constexpr (PMAX == DRX_MAX_MIXED_ORDER)
  {
    switch (orders ? orders[e] : PMAX)   // mixed-order meshes
    {
    case 1: DRX_SPLIT_ELEMENT (1); break;
    case 2: DRX_SPLIT_ELEMENT (2); break;
    case 3: DRX_SPLIT_ELEMENT (3); break;
    default: DRX_SPLIT_ELEMENT (4); break;
    }
  }
  else
    DRX_SPLIT_ELEMENT (PMAX);
#undef DRX_SPLIT_ELEMENT
}

// =============================================================================================
// Bounds reduction (linear_bvh_builder.cpp:19-58)
// =============================================================================================
constexpr int kRedBlock = 256;

__global__ void __launch_bounds__ (kRedBlock) k_bounds_partial (const float *__restrict__ aabbs, int64_t n,
                                                                float *__restrict__ partial)
{
  float mn[3] = { INFINITY, INFINITY, INFINITY }, mx[3] = { -INFINITY, -INFINITY, -INFINITY };
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
  {
    const float *a = aabbs + 6 * i;
#pragma unroll
    for (int d = 0; d < 3; ++d)
    {
      mn[d] = fminf (mn[d], a[2 * d]);
      mx[d] = fmaxf (mx[d], a[2 * d + 1]);
    }
  }
  __shared__ float s[kRedBlock / 64][6];
#pragma unroll
  for (int d = 0; d < 3; ++d)
  {
    mn[d] = wave_reduce_min (mn[d]);
    mx[d] = wave_reduce_max (mx[d]);
  }
  if ((threadIdx.x & 63) == 0)
    for (int d = 0; d < 3; ++d)
    {
      s[threadIdx.x >> 6][2 * d] = mn[d];
      s[threadIdx.x >> 6][2 * d + 1] = mx[d];
    }
  __syncthreads ();
  if (threadIdx.x < 6)
  {
    float v = s[0][threadIdx.x];
    for (int w = 1; w < kRedBlock / 64; ++w)
      v = (threadIdx.x & 1) ? fmaxf (v, s[w][threadIdx.x]) : fminf (v, s[w][threadIdx.x]);
    partial[6 * blockIdx.x + threadIdx.x] = v;
  }
}

// The partial bounds of n_partial blocks -> the bounds (res.include(mins); res.include(maxs), as
// linear_bvh_builder.cpp:49-57) in out[0..5] and the Morton frame (mins, 1 / extent or 0) in out[6..11].
// One block; n_partial 0 leaves the empty box (+inf, -inf).
__global__ void __launch_bounds__ (kRedBlock) k_bounds_final (const float *__restrict__ partial, int n_partial,
                                                              float *__restrict__ out)
{
  __shared__ float s[kRedBlock / 64][6];
  float mn[3] = { INFINITY, INFINITY, INFINITY }, mx[3] = { -INFINITY, -INFINITY, -INFINITY };
  for (int b = threadIdx.x; b < n_partial; b += blockDim.x)
#pragma unroll
    for (int d = 0; d < 3; ++d)
    {
      mn[d] = fminf (mn[d], partial[6 * b + 2 * d]);
      mx[d] = fmaxf (mx[d], partial[6 * b + 2 * d + 1]);
    }
#pragma unroll
  for (int d = 0; d < 3; ++d)
  {
    mn[d] = wave_reduce_min (mn[d]);
    mx[d] = wave_reduce_max (mx[d]);
  }
  if ((threadIdx.x & 63) == 0)
    for (int d = 0; d < 3; ++d)
    {
      s[threadIdx.x >> 6][2 * d] = mn[d];
      s[threadIdx.x >> 6][2 * d + 1] = mx[d];
    }
  __syncthreads ();
  if (threadIdx.x < 3)
  {
    const int d = threadIdx.x;
    float a = s[0][2 * d], b = s[0][2 * d + 1];
    for (int w = 1; w < kRedBlock / 64; ++w)
    {
      a = fminf (a, s[w][2 * d]);
      b = fmaxf (b, s[w][2 * d + 1]);
    }
    float lo = INFINITY, hi = -INFINITY;   // no boxes: the empty box as it stands
    if (n_partial > 0)
    {
      lo = fminf (lo, a);
      hi = fmaxf (hi, a);
      lo = fminf (lo, b);
      hi = fmaxf (hi, b);
    }
    out[2 * d] = lo;
    out[2 * d + 1] = hi;
    const float ext = hi - lo;
    out[6 + d] = lo;
    out[9 + d] = (ext == .0f) ? 0.f : 1.f / ext;
  }
}

// =============================================================================================
// Morton codes (linear_bvh_builder.cpp:60-90, morton_codes.hpp:16-51)
// =============================================================================================
__device__ __forceinline__ uint32_t expand_bits32 (uint32_t x)
{
  x = (x | (x << 16)) & 0x030000FF;
  x = (x | (x << 8)) & 0x0300F00F;
  x = (x | (x << 4)) & 0x030C30C3;
  x = (x | (x << 2)) & 0x09249249;
  return x;
}

__global__ void k_morton (const float *__restrict__ aabbs, int n, const float *__restrict__ frame,
                          uint32_t *__restrict__ keys, int32_t *__restrict__ vals)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float *a = aabbs + 6 * (int64_t)i;
  const float mins[3] = { frame[0], frame[1], frame[2] }, inv[3] = { frame[3], frame[4], frame[5] };
  uint32_t q[3];
#pragma unroll
  for (int d = 0; d < 3; ++d)
  {
    const float lo = a[2 * d], hi = a[2 * d + 1];
    const float c = (lo > hi) ? __builtin_nanf ("") : 0.5f * (lo + hi);
    float x = (c - mins[d]) * inv[d];
    x = fminf (fmaxf (x * 1024.0f, 0.0f), 1023.0f);
    q[d] = (uint32_t)x;
  }
  keys[i] = (expand_bits32 (q[2]) << 2) | (expand_bits32 (q[1]) << 1) | expand_bits32 (q[0]);
  vals[i] = i;
}

// =============================================================================================
// Stable LSD radix sort of (uint32 key, int32 value), 8-bit digits.
// Pass = per-tile histograms -> exclusive scan over (digit, tile) -> stable per-tile scatter.
// =============================================================================================
constexpr int kSortBlock = 256;
constexpr int kSortRounds = 16;
constexpr int kSortTile = kSortBlock * kSortRounds;   // keys per tile

__global__ void __launch_bounds__ (kSortBlock) k_radix_hist (const uint32_t *__restrict__ keys, int n, int shift,
                                                              int n_tiles, int32_t *__restrict__ hist)
{
  __shared__ int32_t h[256];
  h[threadIdx.x] = 0;
  __syncthreads ();
  const int64_t base = (int64_t)blockIdx.x * kSortTile;
  for (int r = 0; r < kSortRounds; ++r)
  {
    const int64_t i = base + r * kSortBlock + threadIdx.x;
    if (i < n) atomicAdd (&h[(keys[i] >> shift) & 0xFF], 1);
  }
  __syncthreads ();
  hist[threadIdx.x * n_tiles + blockIdx.x] = h[threadIdx.x];
}

// Scatter: wavefront w owns the w-th kSortRounds * 64 consecutive keys of its tile.  All its keys are loaded before
// any is ranked (a load per round in front of its ranking made a pass one memory latency per round), its digit
// counts taken with LDS atomics, and after one exchange between the wavefronts it ranks its rounds on its own:
// peers of a round by ballots, the digit's running position in LDS, no block barrier.  A pass
// over 138,567 keys 17.8 -> 7.1 us, over 8.65 M 102 -> 73 us.
__global__ void __launch_bounds__ (kSortBlock) k_radix_scatter (const uint32_t *__restrict__ keys_in,
                                                                 const int32_t *__restrict__ vals_in, int n, int shift,
                                                                 int n_tiles, const int32_t *__restrict__ offs,
                                                                 uint32_t *__restrict__ keys_out,
                                                                 int32_t *__restrict__ vals_out)
{
  constexpr int W = kSortBlock / 64;
  __shared__ int32_t at[W][256];   // per wavefront: digit counts, then the digit's next position
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const uint64_t lt = lanemask_lt ();
  const int64_t base = (int64_t)blockIdx.x * kSortTile + (int64_t)w * (kSortRounds * 64) + lane;
  uint32_t key[kSortRounds];
  int32_t val[kSortRounds];
#pragma unroll
  for (int r = 0; r < kSortRounds; ++r)
  {
    const int64_t i = base + 64 * r;
    key[r] = i < n ? keys_in[i] : 0u;
    val[r] = i < n ? vals_in[i] : 0;
  }
  const int32_t tile_off = offs[(int64_t)threadIdx.x * n_tiles + blockIdx.x];
#pragma unroll
  for (int q = 0; q < W; ++q) at[q][threadIdx.x] = 0;
  __syncthreads ();
#pragma unroll
  for (int r = 0; r < kSortRounds; ++r)
    if (base + 64 * r < n) atomicAdd (&at[w][(key[r] >> shift) & 0xFF], 1);
  __syncthreads ();
  {
    int32_t o = tile_off;   // thread = digit
#pragma unroll
    for (int q = 0; q < W; ++q)
    {
      const int32_t c = at[q][threadIdx.x];
      at[q][threadIdx.x] = o;
      o += c;
    }
  }
  __syncthreads ();
#pragma unroll
  for (int r = 0; r < kSortRounds; ++r)
  {
    const bool valid = base + 64 * r < n;
    const uint32_t digit = (key[r] >> shift) & 0xFF;
    // lanes of this wave with the same digit (invalid lanes form their own group)
    uint64_t peers = __ballot (valid);
    if (!valid) peers = ~peers;
#pragma unroll
    for (int b = 0; b < 8; ++b)
    {
      const uint64_t m = __ballot ((digit >> b) & 1u);
      peers &= ((digit >> b) & 1u) ? m : ~m;
    }
    const int rank = __popcll (peers & lt);
    const int32_t first = at[w][digit];
    __builtin_amdgcn_fence (__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier ();
    if (valid)
    {
      keys_out[first + rank] = key[r];
      vals_out[first + rank] = val[r];
      if (rank == 0) at[w][digit] = first + __popcll (peers);
    }
    __builtin_amdgcn_fence (__ATOMIC_ACQUIRE, "wavefront");
    __builtin_amdgcn_wave_barrier ();
  }
}

// =============================================================================================
// Gathers, Karras tree, refit, emit
// =============================================================================================
__global__ void k_gather_boxes (const int32_t *__restrict__ ids, const float *__restrict__ aabbs,
                                const int32_t *__restrict__ prims, int n, float *__restrict__ s_aabbs,
                                int32_t *__restrict__ leaf_nodes, int32_t *__restrict__ aabb_ids)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t j = ids[i];
#pragma unroll
  for (int q = 0; q < 6; ++q) s_aabbs[6 * (int64_t)i + q] = aabbs[6 * j + q];
  leaf_nodes[i] = prims[j];
  aabb_ids[i] = (int32_t)j;
}

__device__ __forceinline__ int clz_u32 (uint32_t x) { return x == 0 ? 32 : __clz ((int)x); }

__device__ __forceinline__ int karras_delta (int a, int b, int inner_size, const uint32_t *__restrict__ mc)
{
  const bool oor = (b < 0 || b > inner_size);
  const int bb = oor ? 0 : b;
  uint32_t ex = mc[a] ^ mc[bb];
  const bool tie = (ex == 0);
  ex = tie ? ((uint32_t)a ^ (uint32_t)bb) : ex;
  int count = clz_u32 (ex);
  if (tie) count += 32;
  return oor ? -1 : count;
}

// Karras 2012 (linear_bvh_builder.cpp:168-251), including the float ceil of the split search.
__global__ void k_build_tree (const uint32_t *__restrict__ mc, int inner, int32_t *__restrict__ left,
                              int32_t *__restrict__ right, int32_t *__restrict__ parent, int32_t *__restrict__ range_lo,
                              int32_t *__restrict__ range_hi)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= inner) return;
  const int d = 0 > (karras_delta (i, i + 1, inner, mc) - karras_delta (i, i - 1, inner, mc)) ? -1 : 1;
  const int min_delta = karras_delta (i, i - d, inner, mc);
  int lmax = 2;
  while (karras_delta (i, i + lmax * d, inner, mc) > min_delta) lmax *= 2;
  int l = 0;
  for (int t = lmax / 2; t >= 1; t /= 2)
    if (karras_delta (i, i + (l + t) * d, inner, mc) > min_delta) l += t;
  const int j = i + l * d;
  const int delta_node = karras_delta (i, j, inner, mc);
  int s = 0;
  float div = 2.f;
  for (int t = (int)ceilf ((float)l / div);; div *= 2, t = (int)ceilf ((float)l / div))
  {
    if (karras_delta (i, i + (s + t) * d, inner, mc) > delta_node) s += t;
    if (t == 1) break;
  }
  const int split = i + s * d + min (d, 0);
  range_lo[i] = min (i, j);   // node i covers sorted leaves [min(i, j), max(i, j)]
  range_hi[i] = max (i, j);
  if (min (i, j) == split)
  {
    parent[split + inner] = i;
    left[i] = split + inner;
  }
  else
  {
    parent[split] = i;
    left[i] = split;
  }
  if (max (i, j) == split + 1)
  {
    parent[split + inner + 1] = i;
    right[i] = split + inner + 1;
  }
  else
  {
    parent[split + 1] = i;
    right[i] = split + 1;
  }
  if (i == 0) parent[0] = -1;
}

__global__ void k_fill_i32 (int32_t *p, int64_t n, int32_t v)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__device__ __forceinline__ void box_union (float *o, const float *a, const float *b)
{
  // AABB::include of two non-empty ranges per axis (aabb.hpp:46-51): min/max are order independent.
#pragma unroll
  for (int d = 0; d < 3; ++d)
  {
    float lo = INFINITY, hi = -INFINITY;
    if (!(a[2 * d] > a[2 * d + 1]))
    {
      lo = fminf (lo, a[2 * d]);
      hi = fmaxf (hi, a[2 * d]);
      lo = fminf (lo, a[2 * d + 1]);
      hi = fmaxf (hi, a[2 * d + 1]);
    }
    if (!(b[2 * d] > b[2 * d + 1]))
    {
      lo = fminf (lo, b[2 * d]);
      hi = fmaxf (hi, b[2 * d]);
      lo = fminf (lo, b[2 * d + 1]);
      hi = fmaxf (hi, b[2 * d + 1]);
    }
    o[2 * d] = lo;
    o[2 * d + 1] = hi;
  }
}

// propagate_aabbs (linear_bvh_builder.cpp:253-317) without atomics.  A node's box is the exact min/max
// union of the boxes of its contiguous range of sorted leaves (the value propagate_aabbs computes, since
// min/max do not depend on order).  A
// pyramid of pairwise unions over the sorted leaf boxes (level l entry i covers leaves [i 2^l, (i+1) 2^l))
// answers each node's range with at most 2 log2(n) reads, so every node is computed independently.
__device__ __forceinline__ void box_include (float *acc, const float *x)
{
#pragma unroll
  for (int d = 0; d < 3; ++d)
    if (!(x[2 * d] > x[2 * d + 1]))
    {
      acc[2 * d] = fminf (acc[2 * d], x[2 * d]);
      acc[2 * d + 1] = fmaxf (acc[2 * d + 1], x[2 * d]);
      acc[2 * d] = fminf (acc[2 * d], x[2 * d + 1]);
      acc[2 * d + 1] = fmaxf (acc[2 * d + 1], x[2 * d + 1]);
    }
}

constexpr int kMaxLevels = 32;
struct Pyramid
{
  float *level[kMaxLevels];
};

// kPyramidSpan levels per launch: a block reads 2 * kPyramidBlock boxes of level l0 and reduces them pairwise through
// LDS, writing every level on the way.  One launch per level was mostly launch latency (138,567 leaves: 18 launches,
// 41 us; 8.65 M: 24 launches, 240 us); now 13 us
// and 126 us.
constexpr int kPyramidBlock = 256, kPyramidSpan = 9;

__global__ void __launch_bounds__ (kPyramidBlock) k_pyramid_levels (Pyramid pyr, int l0, int n_src)
{
  __shared__ float box[kPyramidBlock][6];
  const int t = threadIdx.x;
  int64_t i = (int64_t)blockIdx.x * kPyramidBlock + t;   // this thread's entry of the level being made
  int n = (n_src + 1) / 2, live = kPyramidBlock;
  float acc[6] = { INFINITY, -INFINITY, INFINITY, -INFINITY, INFINITY, -INFINITY };
  if (i < n)
  {
    const float *src = pyr.level[l0] + 12 * i;
    box_include (acc, src);
    if (2 * i + 1 < n_src) box_include (acc, src + 6);
  }
  for (int l = l0 + 1;; ++l)
  {
    if (t < live && i < n)
    {
      float *dst = pyr.level[l] + 6 * i;
#pragma unroll
      for (int q = 0; q < 6; ++q) dst[q] = box[t][q] = acc[q];
    }
    if (n <= 1 || l == l0 + kPyramidSpan) break;   // block-uniform
    __syncthreads ();
    const int n_below = n;
    n = (n + 1) / 2;
    live >>= 1;
    i = (int64_t)blockIdx.x * live + t;
#pragma unroll
    for (int q = 0; q < 6; ++q) acc[q] = (q & 1) ? -INFINITY : INFINITY;
    if (t < live && i < n)
    {
      box_include (acc, box[2 * t]);
      if (2 * i + 1 < n_below) box_include (acc, box[2 * t + 1]);
    }
    __syncthreads ();
  }
}

__global__ void k_refit_ranges (Pyramid pyr, const int32_t *__restrict__ range_lo, const int32_t *__restrict__ range_hi,
                                int inner, float *__restrict__ inner_aabbs)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= inner) return;
  float acc[6] = { INFINITY, -INFINITY, INFINITY, -INFINITY, INFINITY, -INFINITY };
  int a = range_lo[i], b = range_hi[i] + 1;
  for (int l = 0; a < b; ++l, a >>= 1, b >>= 1)
  {
    if (a & 1) box_include (acc, pyr.level[l] + 6 * (int64_t)(a++));
    if (b & 1) box_include (acc, pyr.level[l] + 6 * (int64_t)(--b));
  }
#pragma unroll
  for (int q = 0; q < 6; ++q) inner_aabbs[6 * (int64_t)i + q] = acc[q];
}

// emit (linear_bvh_builder.cpp:319-397)
__global__ void k_emit (const int32_t *__restrict__ left, const int32_t *__restrict__ right,
                        const float *__restrict__ leaf_aabbs, const float *__restrict__ inner_aabbs, int inner,
                        float4 *__restrict__ out)
{
  const int node = blockIdx.x * blockDim.x + threadIdx.x;
  if (node >= inner) return;
  int lc = left[node], rc = right[node];
  const float *la, *ra;
  if (lc >= inner)
  {
    la = leaf_aabbs + 6 * (int64_t)(lc - inner);
    lc = -(lc - inner + 1);
  }
  else
  {
    la = inner_aabbs + 6 * (int64_t)lc;
    lc *= 4;
  }
  if (rc >= inner)
  {
    ra = leaf_aabbs + 6 * (int64_t)(rc - inner);
    rc = -(rc - inner + 1);
  }
  else
  {
    ra = inner_aabbs + 6 * (int64_t)rc;
    rc *= 4;
  }
  float4 *o = out + 4 * (int64_t)node;
  o[0] = make_float4 (la[0], la[2], la[4], la[1]);
  o[1] = make_float4 (la[3], la[5], ra[0], ra[2]);
  o[2] = make_float4 (ra[4], ra[1], ra[3], ra[5]);
  o[3] = make_float4 (__int_as_float (lc), __int_as_float (rc), 0.f, 0.f);
}

__global__ void k_pack_leaves (const int32_t *__restrict__ leaf_nodes, const int32_t *__restrict__ aabb_ids,
                               const float *__restrict__ subrefs, int n, float4 *__restrict__ out)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float *s = subrefs + 6 * (int64_t)aabb_ids[i];
  out[2 * (int64_t)i] = make_float4 (__int_as_float (leaf_nodes[i]), s[0], s[1], s[2]);
  out[2 * (int64_t)i + 1] = make_float4 (s[3], s[4], s[5], 0.f);
}

static inline unsigned nblk (int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

int radix_tiles (int n) { return (n + kSortTile - 1) / kSortTile; }

int radix_sort_pairs (uint32_t *kA, int32_t *vA, uint32_t *kB, int32_t *vB, int32_t *hist, int n, int bits,
                      hipStream_t st, uint32_t **keys_out, int32_t **vals_out, int32_t *scan_sums)
{
  const int n_tiles = radix_tiles (n);
  uint32_t *ks = kA, *kd = kB;
  int32_t *vs = vA, *vd = vB;
  int32_t *offs = hist + 256 * (size_t)n_tiles;
  for (int shift = 0; shift < bits; shift += 8)
  {
    hipLaunchKernelGGL (k_radix_hist, dim3 (n_tiles), dim3 (kSortBlock), 0, st, ks, n, shift, n_tiles, hist);
    DRX_LAUNCH_CHECK ();
    int rc = exclusive_scan_i32 (hist, offs, 256 * n_tiles, nullptr, st, scan_sums);
    if (rc != DRX_OK) return rc;
    hipLaunchKernelGGL (k_radix_scatter, dim3 (n_tiles), dim3 (kSortBlock), 0, st, ks, vs, n, shift, n_tiles, offs, kd,
                        vd);
    DRX_LAUNCH_CHECK ();
    std::swap (ks, kd);
    std::swap (vs, vd);
  }
  *keys_out = ks;
  *vals_out = vs;
  return DRX_OK;
}

// Morton codes of query points in the normalised frame of `bounds` (the LBVH's 30-bit quantisation),
// kept to their top kPointMortonBits bits: the order only groups nearby points for coherent walks (any
// order gives the same results), and 24 bits (256 cells per axis) sort in three radix passes, not four.
#ifndef DRX_POINT_MORTON_BITS
#define DRX_POINT_MORTON_BITS 24
#endif
constexpr int kPointMortonBits = DRX_POINT_MORTON_BITS;

__global__ void k_point_morton (const float *__restrict__ pts, int n, float minx, float miny, float minz, float ix,
                                float iy, float iz, uint32_t *__restrict__ keys, int32_t *__restrict__ vals)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float mins[3] = { minx, miny, minz }, inv[3] = { ix, iy, iz };
  uint32_t q[3];
#pragma unroll
  for (int d = 0; d < 3; ++d)
  {
    float x = (pts[3 * (int64_t)i + d] - mins[d]) * inv[d];
    x = fminf (fmaxf (x * 1024.0f, 0.0f), 1023.0f);
    q[d] = (uint32_t)x;
  }
  keys[i] = ((expand_bits32 (q[2]) << 2) | (expand_bits32 (q[1]) << 1) | expand_bits32 (q[0])) >> (30 - kPointMortonBits);
  vals[i] = i;
}

int sort_scratch (int n, hipStream_t st, SortScratch *out)
{
  out->kA = (uint32_t *)arena (SLOT_SORT_KEYS_A, sizeof (uint32_t) * (size_t)n, st);
  out->kB = out->kA ? (uint32_t *)arena (SLOT_SORT_KEYS_B, sizeof (uint32_t) * (size_t)n, st) : nullptr;
  out->vA = out->kB ? (int32_t *)arena (SLOT_SORT_VALS_A, sizeof (int32_t) * (size_t)n, st) : nullptr;
  out->vB = out->vA ? (int32_t *)arena (SLOT_SORT_VALS_B, sizeof (int32_t) * (size_t)n, st) : nullptr;
  out->hist = out->vB ? (int32_t *)arena (SLOT_SORT_HIST, sizeof (int32_t) * (size_t)radix_hist_len (n), st) : nullptr;
  out->scan_sums = out->hist ? (int32_t *)arena (SLOT_SCAN, sizeof (int32_t) * (size_t)scan_sums_len (256 * radix_tiles (n)), st)
                             : nullptr;
  return out->scan_sums ? DRX_OK : DRX_ERR_HIP;
}

void sort_scratch_free (hipStream_t st)
{
  for (int s : { SLOT_SORT_KEYS_A, SLOT_SORT_KEYS_B, SLOT_SORT_VALS_A, SLOT_SORT_VALS_B, SLOT_SORT_HIST }) arena_free (s, st);
}

int morton_order_points (const float *pts, int n, const float *bounds6, hipStream_t st, const int32_t **order_out,
                         const SortScratch &ws)
{
  float minc[3], inv[3];
  for (int d = 0; d < 3; ++d)
  {
    minc[d] = bounds6[2 * d];
    const float ext = bounds6[2 * d + 1] - bounds6[2 * d];
    inv[d] = (ext > 0.f) ? 1.f / ext : 0.f;
  }
  hipLaunchKernelGGL (k_point_morton, dim3 (nblk (n, 256)), dim3 (256), 0, st, pts, n, minc[0], minc[1], minc[2], inv[0],
                      inv[1], inv[2], ws.kA, ws.vA);
  DRX_LAUNCH_CHECK ();
  uint32_t *ks;
  int32_t *vs;
  int rc = radix_sort_pairs (ws.kA, ws.vA, ws.kB, ws.vB, ws.hist, n, kPointMortonBits, st, &ks, &vs, ws.scan_sums);
  if (rc) return rc;
  *order_out = vs;
  return DRX_OK;
}

} // namespace drx

using namespace drx;

extern "C" {

int drx_bvh_split_elements (const int32_t *ctrl_idx, const float *values, const int32_t *orders, const int64_t *offsets,
                            int32_t order, int32_t n_el, float *out_aabbs, int32_t *out_prims, float *out_subrefs,
                            void *stream)
{
  if (n_el < 0) return fail (DRX_ERR_ARG, "drx_bvh_split_elements: n_el < 0");
  if (n_el == 0) return DRX_OK;
  if (!ctrl_idx || !values || !out_aabbs || !out_prims || !out_subrefs)
    return fail (DRX_ERR_ARG, "drx_bvh_split_elements: null pointer");
  if ((orders == nullptr) != (offsets == nullptr))
    return fail (DRX_ERR_ARG, "drx_bvh_split_elements: orders and offsets go together");
  const int pmax = orders ? DRX_MAX_MIXED_ORDER : order;
  if (pmax < 1 || pmax > DRX_MAX_ORDER)
    return fail (DRX_ERR_ARG, "drx_bvh_split_elements: order %d outside 1..%d", order, DRX_MAX_ORDER);
  hipStream_t st = as_stream (stream);
#define DRX_SPLIT_GO(P, W)                                                                                       \
  hipLaunchKernelGGL ((k_split<P, W>), dim3 (n_el), dim3 (64 * W), 0, st, ctrl_idx, values, orders, offsets, n_el, \
                      out_aabbs, out_prims, out_subrefs)
  switch (pmax)
  {
  // wavefronts per element: order 2 one (64,000 elements 249 us, two 260), order 3 four (262,144 elements
  // 1.08 ms, two 1.15, one 1.31), order 4 four (64,000 elements 672 us, two 789)
  case 1: DRX_SPLIT_GO (1, 1); break;
  case 2: DRX_SPLIT_GO (2, 1); break;
  case 3: DRX_SPLIT_GO (3, 4); break;
  case 4: DRX_SPLIT_GO (4, 4); break;
  case 5: DRX_SPLIT_GO (5, 4); break;
  case 6: DRX_SPLIT_GO (6, 8); break;
  case 7: DRX_SPLIT_GO (7, 8); break;
  default: DRX_SPLIT_GO (8, 8); break;
  }
#undef DRX_SPLIT_GO
  DRX_LAUNCH_CHECK ();
  return DRX_OK;
}

int drx_bvh_build (const float *aabbs_in, const int32_t *prims_in, int32_t n_in, float *out_inner,
                   int32_t *out_leaf_nodes, int32_t *out_aabb_ids, float *out_bounds, uint32_t *out_mcodes,
                   void *stream)
{
  if (n_in < 0) return fail (DRX_ERR_ARG, "drx_bvh_build: n < 0");
  if (!out_inner || !out_leaf_nodes || !out_aabb_ids || !out_bounds)
    return fail (DRX_ERR_ARG, "drx_bvh_build: null output");
  if (n_in > 0 && (!aabbs_in || !prims_in)) return fail (DRX_ERR_ARG, "drx_bvh_build: null input");
  if (n_in > (1 << 30)) return fail (DRX_ERR_ARG, "drx_bvh_build: %d boxes exceed the int32 tree index range", n_in);
  hipStream_t st = as_stream (stream);
  const float *aabbs = aabbs_in;
  const int32_t *prims = prims_in;
  const bool zero_case = (n_in == 0);
  const int n = n_in < 2 ? 2 : n_in;
  // dray pads 0 and 1 boxes to two (linear_bvh_builder.cpp:411-456)
  float hb[12] = { 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0 };
  int32_t hp[2] = { 0, 0 };
  if (n_in < 2)
  {
    if (n_in == 1)
    {
      DRX_HIP (hipMemcpyAsync (hb, aabbs_in, 6 * sizeof (float), hipMemcpyDeviceToHost, st));
      DRX_HIP (hipMemcpyAsync (hp, prims_in, sizeof (int32_t), hipMemcpyDeviceToHost, st));
      DRX_HIP (hipStreamSynchronize (st));
      hp[1] = hp[0];
    }
    float *pa = (float *)arena (SLOT_TREE2, 12 * sizeof (float) + 2 * sizeof (int32_t), st);
    if (!pa) return DRX_ERR_HIP;
    DRX_HIP (hipMemcpyAsync (pa, hb, 12 * sizeof (float), hipMemcpyHostToDevice, st));
    DRX_HIP (hipMemcpyAsync (pa + 12, hp, 2 * sizeof (int32_t), hipMemcpyHostToDevice, st));
    DRX_HIP (hipStreamSynchronize (st));
    aabbs = pa;
    prims = (const int32_t *)(pa + 12);
  }
  const int inner = n - 1;
  // scratch: keys/vals ping-pong, histogram, tree arrays
  const int n_tiles = (n + kSortTile - 1) / kSortTile;
  uint32_t *kA = (uint32_t *)arena (SLOT_SORT_KEYS_A, sizeof (uint32_t) * n, st);
  uint32_t *kB = (uint32_t *)arena (SLOT_SORT_KEYS_B, sizeof (uint32_t) * n, st);
  int32_t *vA = (int32_t *)arena (SLOT_SORT_VALS_A, sizeof (int32_t) * n, st);
  int32_t *vB = (int32_t *)arena (SLOT_SORT_VALS_B, sizeof (int32_t) * n, st);
  int32_t *hist = (int32_t *)arena (SLOT_SORT_HIST, sizeof (int32_t) * (2 * 256 * (size_t)n_tiles + 8), st);
  // tree slot: sorted aabbs (6n) | inner aabbs (6 inner) | left | right | parent (2n-1) | partial bounds
  const int red_blocks = std::min (1024, (int)nblk (n, kRedBlock));
  const size_t tree_floats = 6 * (size_t)n + 6 * (size_t)inner;
  const size_t tree_ints = (size_t)inner * 2 + (2 * (size_t)n - 1);
  char *tree = (char *)arena (SLOT_TREE, tree_floats * 4 + tree_ints * 4 + 6 * 4 * (size_t)red_blocks + 128, st);
  if (!kA || !kB || !vA || !vB || !hist || !tree) return DRX_ERR_HIP;
  float *s_aabbs = (float *)tree;
  float *i_aabbs = s_aabbs + 6 * (size_t)n;
  int32_t *left = (int32_t *)(i_aabbs + 6 * (size_t)inner);
  int32_t *right = left + inner;
  int32_t *parent = right + inner;
  float *partial = (float *)(parent + (2 * (size_t)n - 1));

  // bounds, reduced on the device (no host round trip before the Morton codes); copied out at the end
  float *dbounds = partial + 6 * (size_t)red_blocks;   // bounds[6], Morton frame (mins, 1 / extent)[6]
  if (!zero_case)
  {
    hipLaunchKernelGGL (k_bounds_partial, dim3 (red_blocks), dim3 (kRedBlock), 0, st, aabbs, (int64_t)n, partial);
    DRX_LAUNCH_CHECK ();
  }
  hipLaunchKernelGGL (k_bounds_final, dim3 (1), dim3 (kRedBlock), 0, st, partial, zero_case ? 0 : red_blocks, dbounds);
  DRX_LAUNCH_CHECK ();
  hipLaunchKernelGGL (k_morton, dim3 (nblk (n, 256)), dim3 (256), 0, st, aabbs, n, dbounds + 6, kA, vA);
  DRX_LAUNCH_CHECK ();
  // stable radix sort, 8-bit digits over 30-bit keys
  uint32_t *ks = nullptr;
  int32_t *vs = nullptr;
  {
    int rc = radix_sort_pairs (kA, vA, kB, vB, hist, n, 30, st, &ks, &vs);
    if (rc != DRX_OK) return rc;
  }
  // ks = sorted codes, vs = ids
  if (out_mcodes) DRX_HIP (hipMemcpyAsync (out_mcodes, ks, sizeof (uint32_t) * n, hipMemcpyDeviceToDevice, st));
  hipLaunchKernelGGL (k_gather_boxes, dim3 (nblk (n, 256)), dim3 (256), 0, st, vs, aabbs, prims, n, s_aabbs,
                      out_leaf_nodes, out_aabb_ids);
  DRX_LAUNCH_CHECK ();
  // pyramid levels 1.. over the sorted leaf boxes (level 0), plus the node ranges
  size_t pyr_floats = 0;
  int n_levels = 1;
  for (int64_t m = n; m > 1; m = (m + 1) / 2)
  {
    pyr_floats += 6 * (size_t)((m + 1) / 2);
    ++n_levels;
  }
  if (n_levels > kMaxLevels) return fail (DRX_ERR_ARG, "drx_bvh_build: too many boxes for the refit pyramid");
  char *pyr_mem = (char *)arena (SLOT_PYRAMID, pyr_floats * sizeof (float) + 2 * sizeof (int32_t) * (size_t)inner + 64, st);
  if (!pyr_mem) return DRX_ERR_HIP;
  int32_t *range_lo = (int32_t *)pyr_mem;
  int32_t *range_hi = range_lo + inner;
  float *levels = (float *)(range_hi + inner);
  hipLaunchKernelGGL (k_build_tree, dim3 (nblk (inner, 256)), dim3 (256), 0, st, ks, inner, left, right, parent,
                      range_lo, range_hi);
  Pyramid pyr;
  pyr.level[0] = s_aabbs;
  {
    int sizes[kMaxLevels] = { n };
    for (int l = 1; l < kMaxLevels; ++l)
    {
      pyr.level[l] = l < n_levels ? levels : nullptr;
      sizes[l] = (sizes[l - 1] + 1) / 2;
      if (l < n_levels) levels += 6 * (size_t)sizes[l];
    }
    for (int l = 0; l < n_levels - 1; l += kPyramidSpan)
      hipLaunchKernelGGL (k_pyramid_levels, dim3 (nblk (sizes[l], 2 * kPyramidBlock)), dim3 (kPyramidBlock), 0, st, pyr, l,
                          sizes[l]);
  }
  hipLaunchKernelGGL (k_refit_ranges, dim3 (nblk (inner, 256)), dim3 (256), 0, st, pyr, range_lo, range_hi, inner, i_aabbs);
  hipLaunchKernelGGL (k_emit, dim3 (nblk (inner, 256)), dim3 (256), 0, st, left, right, s_aabbs, i_aabbs, inner,
                      (float4 *)out_inner);
  DRX_LAUNCH_CHECK ();
  return read_back (out_bounds, dbounds, 6 * sizeof (float), st);
}

int drx_bvh_pack_leaves (const drx_bvh *bvh, float *out_leaf_pack, void *stream)
{
  if (!bvh || !out_leaf_pack || !bvh->leaf_nodes || !bvh->aabb_ids || !bvh->subrefs)
    return fail (DRX_ERR_ARG, "drx_bvh_pack_leaves: null pointer");
  hipLaunchKernelGGL (k_pack_leaves, dim3 (nblk (bvh->n_leaves, 256)), dim3 (256), 0, as_stream (stream), bvh->leaf_nodes,
                      bvh->aabb_ids, bvh->subrefs, bvh->n_leaves, (float4 *)out_leaf_pack);
  DRX_LAUNCH_CHECK ();
  return DRX_OK;
}

} // extern "C"
