// Point location for a workgroup's batch of points with the candidates binned by element.
//
// With one lane per point a wavefront's lanes test their candidates together, each reading the control points of
// its own element: at order 3 a Newton step is 48 16-byte reads per lane, and the vector-memory data path, not the
// arithmetic, bounds it (30 to 46 cycles per wavefront read; four SIMDs share it).  Here a workgroup takes up
// to N points that lie close together (consecutive samples of neighbouring rays):
//   1. each wavefront collects the leaves that the box around its points overlaps, by one cooperative descent of
//      the compact nodes, a lane per frontier node, in depth-first order; its points are then tested against those
//      leaves' exact boxes by broadcast LDS reads (where the leaves are too many, each lane walks by itself);
//   2. the points are grouped by candidate element in a small LDS hash table;
//   3. whole wavefronts are given to one element at a time: its control points come in by scalar loads and feed the
//      multiply-adds as scalar operands; elements with few points share wavefronts that read per lane;
//   4. rejected points go round again with their next candidate.
// A point sees the candidates of its own depth-first walk in the same order, with the same arithmetic, whatever it
// shares a wavefront with.
#pragma once

#include "drx_element.hpp"
#include "drx_wave.hpp"

namespace drx
{

constexpr int kBinThreads = 256, kBinWaves = kBinThreads / 64;
constexpr int kBinSlots = kBinThreads;       // hash slots, one per thread in the prefix sum
// Points from which an element gets wavefronts of its own.  A task for one element leaves lanes idle, one for several
// reads control points per lane: 4 / 8 / 12 / 24 / 32 / 48 points give 10.5 / 9.9 / 9.5 / 9.29 / 9.28 / 9.27 ms on
// the 64^3 order-3 frame and 58.7 / 57.2 / 53.4 / 51.6 / 51.6 / 52.6 ms on the 40^3 order-4 frame (1024^2 rays, 512
// samples; 1000^2, 1000).
constexpr int kBinMin = 32;
// Leaves a wavefront's list holds.  112 let four blocks share a CU's LDS; with 224 two do (order-3 frame 12.7 ms
// against 9.4 ms).
constexpr int kBinLeaves = 112;
constexpr int kBinProbes = 8;
typedef TravStackOf<0> BinStack;              // of a lane that walks by itself (rare): no LDS
// A point that has tried this many candidates is left: it is not for this form, where a round of few points leaves most of the
// block idle and a point that walks by itself starts its walk anew in every round.
constexpr int kBinCands = 128;
// A point's record: Newton steps (17 bits), candidates (12 bits), flags.
constexpr uint32_t kRecSteps = (1u << 17) - 1, kRecCandOne = 1u << 17, kRecCands = 0xFFFu << 17, kRecOverflow = 1u << 29,
                   kRecFound = 1u << 30, kRecPolished = 1u << 31;
// What follows a point's candidate: a leaf (>= 0), nothing, a candidate that only a walk finds, or an entry of a
// wavefront's list (wavefront * kBinLeaves + entry) that is the next hit (kNextMore: hits follow it) or after which
// to look on for one (kNextScan).
constexpr int32_t kNextNone = -1, kNextWalk = -2, kNextList = -16;   // kNextList - (entry | flags)
constexpr int32_t kNextMore = 1 << 12, kNextScan = 1 << 13, kNextEntry = (1 << 12) - 1;
constexpr int32_t kLeafMore = 1 << 30;   // on a leaf: further hits, found by a walk
static_assert (kBinWaves * kBinLeaves <= kNextEntry, "list entries fit their bits");
static_assert (kBinCands <= (int)(kRecCands / kRecCandOne) && kBinCands * 20 <= (int)kRecSteps, "counts fit their bits");

// A leaf of a wavefront's list: exact box, element and leaf index.
struct BinLeaf
{
  float lx, ly, lz, hx, hy, hz;
  int32_t el, leaf;
};
static_assert (sizeof (BinLeaf) == 32, "two 16-byte LDS reads");

// One wavefront's memory for finding candidates.
union BinWave
{
  int32_t front[2][kBinLeaves];      // the descent's frontiers, then
  BinLeaf list[kBinLeaves + 1];      // its leaves (the last entry is never hit)
};

template <int N> struct BinShared
{
  BinWave wave[kBinWaves];
  union
  {
    int32_t top[kBinWaves][kBinLeaves];   // finding candidates: the frontier at which a descent outgrew the list
    uint16_t group[N];                    // testing them: the points grouped by element
  };
  int32_t leaf[N], after[N];   // each point's candidate and what follows it
  uint32_t rec[N];
  uint16_t next[N];  // rejected points
  int32_t key[kBinSlots], num[kBinSlots + 1];   // element and point count per slot; slot kBinSlots: no slot found
  uint16_t base[kBinSlots + 1];
  uint32_t work[2 * (N / 64) + N / kBinMin + 2];   // wavefront tasks: start | points << 10 | one element << 31
  int32_t wsum[kBinWaves], n_leaves[kBinWaves], n_next, n_work, take;
};

__device__ __forceinline__ void bin_wave_sync ()
{
  __builtin_amdgcn_fence (__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier ();
  __builtin_amdgcn_fence (__ATOMIC_ACQUIRE, "wavefront");
}

// One wavefront's descent from the n codes of front[0] (in depth-first order): the leaves whose cell ranges overlap
// [lo, hi] (wave-uniform grid cells), in depth-first order, into the list; their number.  Where the frontier outgrows
// the list: -1, and with top the frontier before that (n_top codes).
__device__ __forceinline__ int bin_descend (const LocateCfg &cfg, const int lo[3], const int hi[3], BinWave &mem, int n,
                                            int32_t *top, int &n_top, int lane)
{
  int32_t (*front)[kBinLeaves] = mem.front;
  BinLeaf *list = mem.list;
  const uint64_t lt = lanemask_lt ();
  int from = 0;
  for (;;)
  {
    int m = 0;
    bool deeper = false;
    for (int c = 0; c < n; c += 64)
    {
      const bool have = c + lane < n;
      const int code = have ? front[from][c + lane] : -1;
      const bool inner = code >= 0;
      bool in_l = have, in_r = false;   // a leaf stays
      int l = code, r = 0;
      if (inner)
      {
        const uint4 A = cfg.qnodes[code], B = cfg.qnodes[code + 1];
        in_l = lo[0] <= (int)(A.y >> 16) && lo[1] <= (int)(A.z & 0xFFFFu) && lo[2] <= (int)(A.z >> 16) &&
               hi[0] >= (int)(A.x & 0xFFFFu) && hi[1] >= (int)(A.x >> 16) && hi[2] >= (int)(A.y & 0xFFFFu);
        in_r = lo[0] <= (int)(B.x >> 16) && lo[1] <= (int)(B.y & 0xFFFFu) && lo[2] <= (int)(B.y >> 16) &&
               hi[0] >= (int)(A.w & 0xFFFFu) && hi[1] >= (int)(A.w >> 16) && hi[2] >= (int)(B.x & 0xFFFFu);
        l = (int)B.z;
        r = (int)B.w;
      }
      const uint64_t bl = __ballot (in_l), br = __ballot (in_r);
      if (m + __popcll (bl) + __popcll (br) > kBinLeaves)
      {
        if (top)
        {
          for (int u = lane; u < n; u += 64) top[u] = front[from][u];
          n_top = n;
          bin_wave_sync ();
        }
        return -1;
      }
      const int at = m + __popcll (bl & lt) + __popcll (br & lt);
      if (in_l) front[from ^ 1][at] = l;
      if (in_r) front[from ^ 1][at + (in_l ? 1 : 0)] = r;
      m += __popcll (bl) + __popcll (br);
      deeper = deeper || __ballot (inner) != 0;
    }
    bin_wave_sync ();
    from ^= 1;
    n = m;
    if (!deeper) break;
  }
  // the leaves' records replace the frontiers
  constexpr int C = (kBinLeaves + 63) / 64;
  int leaf[C];
#pragma unroll
  for (int c = 0; c < C; ++c) leaf[c] = 64 * c + lane < n ? -front[from][64 * c + lane] - 1 : -1;
  bin_wave_sync ();
#pragma unroll
  for (int c = 0; c < C; ++c)
    if (leaf[c] >= 0)
    {
      const float4 b0 = cfg.leaf_boxes[2 * (int64_t)leaf[c]], b1 = cfg.leaf_boxes[2 * (int64_t)leaf[c] + 1];
      list[64 * c + lane] = BinLeaf { b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, __float_as_int (cfg.leaves[2 * (int64_t)leaf[c]].x),
                                      leaf[c] };
    }
  if (lane == 0) list[kBinLeaves] = BinLeaf { INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY, -1, -1 };
  bin_wave_sync ();
  return n;
}

// dray's inclusive point-in-box test (a NaN coordinate is in no box).
__device__ __forceinline__ bool bin_inside (const BinLeaf &b, const float pt[3])
{
  return pt[0] >= b.lx && pt[1] >= b.ly && pt[2] >= b.lz && pt[0] <= b.hx && pt[1] <= b.hy && pt[2] <= b.hz;
}

// The wavefront's 64 points (NaN: none) against its list of n leaves: list entries of the first two hits (-1: none) and
// whether there are more.
__device__ __forceinline__ void bin_hits (const BinLeaf *list, int n, const float pt[3], int lane, int &first, int &second,
                                          bool &more)
{
  // the leaves that the box around the points overlaps
  float lo[3], hi[3];
#pragma unroll
  for (int d = 0; d < 3; ++d)
  {
    lo[d] = wave_reduce_min (pt[d]);
    hi[d] = wave_reduce_max (pt[d]);
  }
  first = second = -1;
  more = false;
  for (int c = 0; c < n; c += 64)
  {
    bool near_ = false;
    if (c + lane < n)
    {
      const BinLeaf b = list[c + lane];
      near_ = hi[0] >= b.lx && hi[1] >= b.ly && hi[2] >= b.lz && lo[0] <= b.hx && lo[1] <= b.hy && lo[2] <= b.hz;
    }
    uint64_t todo = __ballot (near_);
    while (todo)
    {
      int j[4];
#pragma unroll
      for (int u = 0; u < 4; ++u)
      {
        j[u] = todo ? c + __ffsll ((unsigned long long)todo) - 1 : kBinLeaves;
        todo &= todo - 1;   // 0 stays 0
      }
      BinLeaf b[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) b[u] = list[j[u]];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (bin_inside (b[u], pt))
        {
          more = more || second >= 0;
          second = first >= 0 && second < 0 ? j[u] : second;
          first = first < 0 ? j[u] : first;
        }
    }
  }
}

// Locates the points of a workgroup (all threads call it; Q = N / kBinThreads points per thread: items
// (wavefront * Q + q) * 64 + lane).
//   own_point (q, pt): whether this thread's q-th point is to be located, and its coordinates;
//   point (item, pt): any item's coordinates;
//   accept (item, el, ref, uni): called by one lane for a located item (uni: std::true_type when el is uniform);
//   span: sets of 64 points per leaf list where one list cannot hold those of all sets (Q / 2 at first, halved when
//   a list overflows, kept by the caller between calls).
// Leaves sh.rec[item] (with kBinCands candidates and not found: perhaps unfinished); ends with a barrier.
template <int P, bool POLISH, int N, typename OwnPoint, typename Point, typename Accept>
__device__ __forceinline__ void locate_binned (const LocateCfg &cfg, BinShared<N> &sh, int &span, OwnPoint &&own_point,
                                               Point &&point, Accept &&accept)
{
  constexpr int Q = N / kBinThreads;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  BinStack todo;
  sh.key[tid] = -1;
  sh.num[tid] = 0;
  if (tid == 0) sh.num[kBinSlots] = 0;
  int n_leaves = -1, sets = Q, n_top = 0;
  __syncthreads ();   // the cleared table
  int n_list = N;
  for (int round = 0;; ++round)
  {
    // find the next candidate; enter its element's slot
    uint32_t place[Q];   // item | slot << 10 | rank << 19, or ~0
#pragma unroll
    for (int q = 0; q < Q; ++q) place[q] = ~0u;
#pragma unroll 1
    for (int q = 0; q < Q; ++q)
    {
      const int k = (wv * Q + q) * 64 + lane;
      if (round && (wv * Q + q) * 64 >= n_list) break;   // wave-uniform
      uint32_t mine = ~0u;
      int item = k, el = -1, leaf = -1, after = kNextNone;
      float pt[3] = { 0.f, 0.f, 0.f };
      bool walk = false;
      if (!round)
      {
        while (cfg.qnodes && (q & (sets - 1)) == 0)
        {
          // the leaves that the next `sets` sets of points can be in: all of them from the root; where those outgrow the
          // list, fewer at a time from the frontier reached then
          int lo[3] = { 65535, 65535, 65535 }, hi[3] = { 0, 0, 0 };
          for (int u = q; u < q + sets; ++u)
            if (own_point (u, pt))
#pragma unroll
              for (int d = 0; d < 3; ++d)
              {
                const int c = (int)grid_cell (pt[d], cfg.q_org[d], cfg.q_inv[d]);
                lo[d] = min (lo[d], c);
                hi[d] = max (hi[d], c);
              }
#pragma unroll
          for (int d = 0; d < 3; ++d)
          {
            lo[d] = wave_reduce_min (lo[d]);
            hi[d] = wave_reduce_max (hi[d]);
          }
          const bool all = sets == Q;
          if (all)
          {
            if (lane == 0) sh.wave[wv].front[0][0] = 0;
          }
          else
            for (int u = lane; u < n_top; u += 64) sh.wave[wv].front[0][u] = sh.top[wv][u];
          bin_wave_sync ();
          n_leaves = lo[0] <= hi[0] ? bin_descend (cfg, lo, hi, sh.wave[wv], all ? 1 : n_top, all ? sh.top[wv] : nullptr,
                                                   n_top, lane) : 0;
          if (n_leaves >= 0 || sets == 1) break;
          if (!all) span >>= 1;
          sets = span;
        }
        const bool act = own_point (q, pt);
        if (!act) pt[0] = __builtin_nanf ("");
        sh.rec[k] = 0;
        if (n_leaves >= 0)
        {
          const BinLeaf *list = sh.wave[wv].list;
          int first, second;
          bool more;
          bin_hits (list, n_leaves, pt, lane, first, second, more);
          if (first >= 0)
          {
            leaf = list[first].leaf;
            el = list[first].el;
            if (second >= 0)
              after = sets == Q ? kNextList - ((wv * kBinLeaves + second) | (more ? kNextMore : 0))   // the list stays
                                : list[second].leaf | (more ? kLeafMore : 0);
          }
          if (sets == Q)
          {
            if (lane == 0) sh.n_leaves[wv] = n_leaves;
          }
          else
            bin_wave_sync ();   // the next list's frontiers may replace this one
        }
        else
          walk = act;
      }
      else if (k < n_list)
      {
        item = sh.next[k];
        const int32_t a = sh.after[item];
        if (a >= 0)
        {
          leaf = a & ~kLeafMore;
          after = (a & kLeafMore) ? kNextWalk : kNextNone;
          el = __float_as_int (cfg.leaves[2 * (int64_t)leaf].x);
        }
        else if (a <= kNextList)
        {
          const int32_t f = kNextList - a;
          const int w = (f & kNextEntry) / kBinLeaves;
          int j = (f & kNextEntry) % kBinLeaves;
          const BinLeaf *list = sh.wave[w].list;
          bool hit = true;
          if (f & kNextScan)
          {
            point (item, pt);
            const int n = sh.n_leaves[w];
            do
              ++j;
            while (j < n && !bin_inside (list[j], pt));
            hit = j < n;
          }
          if (hit)
          {
            leaf = list[j].leaf;
            el = list[j].el;
            after = (f & (kNextMore | kNextScan)) ? kNextList - ((w * kBinLeaves + j) | kNextScan) : kNextNone;
          }
        }
        else
          walk = a == kNextWalk;
        if (walk) point (item, pt);
      }
      if (walk)
      {
        int tried = round;   // an item in round r has tried r candidates
        int cur, sp;
        float4 l0, l1, map[3];
        walk_start (cfg, todo, pt, cur, sp);
        for (;;)
        {
          leaf = next_candidate_leaf (cfg, todo, pt, cur, sp, l0, l1, map);
          if (leaf < 0 || tried-- == 0) break;
          cur = todo.get (sp);
          --sp;
        }
        if (leaf == kWalkOverflow) sh.rec[item] |= kRecOverflow;
        if (leaf >= 0) el = __float_as_int (l0.x);
        after = kNextWalk;
      }
      if (leaf >= 0)
      {
        sh.leaf[item] = leaf;
        sh.after[item] = after;
        int slot = kBinSlots, h = (int)(((uint32_t)el * 0x9E3779B1u) >> 24);
#pragma unroll 1
        for (int t = 0; t < kBinProbes; ++t)
        {
          const int32_t was = atomicCAS (&sh.key[h], -1, el);
          if (was == -1 || was == el)
          {
            slot = h;
            break;
          }
          h = (h + 1) & (kBinSlots - 1);
        }
        const int rank = atomicAdd (&sh.num[slot], 1);
        mine = (uint32_t)item | ((uint32_t)slot << 10) | ((uint32_t)rank << 19);
      }
#pragma unroll
      for (int t = 0; t < Q; ++t) place[t] = t == q ? mine : place[t];
    }
    __syncthreads ();
    // places: elements with wavefronts of their own first, then the others; one prefix sum of packed counts
    // (points of own elements | their tasks << 11 | other points << 21)
    const int num = sh.num[tid];
    const bool own = num >= kBinMin;
    const int32_t v = own ? num | (((num + 63) >> 6) << 11) : (int32_t)((uint32_t)num << 21);
    const int32_t incl = wave_scan_incl_add (v);
    if (lane == 63) sh.wsum[wv] = incl;
    __syncthreads ();
    int32_t before = incl - v, total = 0;
#pragma unroll
    for (int q = 0; q < kBinWaves; ++q)
    {
      before += q < wv ? sh.wsum[q] : 0;
      total += sh.wsum[q];
    }
    const int n_own = total & 0x7FF, t_own = (total >> 11) & 0x3FF, n_other = (int)((uint32_t)total >> 21) + sh.num[kBinSlots];
    {
      const int start = own ? before & 0x7FF : n_own + (int)((uint32_t)before >> 21);
      sh.base[tid] = (uint16_t)start;
      if (own)
        for (int t = 0; 64 * t < num; ++t)
          sh.work[((before >> 11) & 0x3FF) + t] = (uint32_t)(start + 64 * t) | ((uint32_t)min (64, num - 64 * t) << 10) |
                                                  0x80000000u;
      const int t_other = (n_other + 63) >> 6;
      if (tid < t_other)
        sh.work[t_own + tid] = (uint32_t)(n_own + 64 * tid) | ((uint32_t)min (64, n_other - 64 * tid) << 10);
      if (tid == 0)
      {
        sh.base[kBinSlots] = (uint16_t)(n_own + n_other - sh.num[kBinSlots]);
        sh.n_work = t_own + t_other;
        sh.n_next = 0;
        sh.take = 0;
      }
    }
    __syncthreads ();
#pragma unroll
    for (int q = 0; q < Q; ++q)
      if (place[q] != ~0u)
        sh.group[sh.base[(place[q] >> 10) & 0x1FF] + (place[q] >> 19)] = (uint16_t)(place[q] & 0x3FF);
    __syncthreads ();
    // test the candidates, one task per wavefront at a time
    const int n_work = sh.n_work;
    for (;;)
    {
      int t = 0;
      if (lane == 0) t = atomicAdd (&sh.take, 1);
      t = __builtin_amdgcn_readfirstlane (t);
      if (t >= n_work) break;
      const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane ((int)sh.work[t]);
      if (lane < (int)((w >> 10) & 0x7F))
      {
        const int item = sh.group[(w & 0x3FF) + lane];
        const int leaf = sh.leaf[item];
        const float4 l0 = cfg.leaves[2 * (int64_t)leaf], l1 = cfg.leaves[2 * (int64_t)leaf + 1];
        float pt[3], x[3];
        point (item, pt);
        candidate_start<P> (cfg, __float_as_int (l0.x), leaf, pt, l0, l1, x);
        LocateStats st { 0, 0, 0, 0 };
        bool found;
        if (w >> 31)
        {
          const int el = __builtin_amdgcn_readfirstlane (__float_as_int (l0.x));   // the same in every lane
          if constexpr (P == 0)
            found = try_element_mixed<POLISH, true> (cfg, el, pt, x, st);
          else
            found = try_element_at<P, POLISH, true> (cfg, cfg.mesh + (int64_t)el * Ord<P>::GSTRIDE, pt, x, st);
          if (found) accept (item, el, x, std::true_type ());
        }
        else
        {
          const int el = __float_as_int (l0.x);
          if constexpr (P == 0)
            found = try_element_mixed<POLISH> (cfg, el, pt, x, st);
          else
            found = try_element_at<P, POLISH> (cfg, cfg.mesh + (int64_t)el * Ord<P>::GSTRIDE, pt, x, st);
          if (found) accept (item, el, x, std::false_type ());
        }
        uint32_t c = sh.rec[item];
        c += kRecCandOne + (uint32_t)st.newton;
        sh.rec[item] = c | (found ? kRecFound : 0) | (st.polished ? kRecPolished : 0);
        if (!found && (c & kRecCands) < kBinCands * kRecCandOne) sh.next[atomicAdd (&sh.n_next, 1)] = (uint16_t)item;
      }
    }
    sh.key[tid] = -1;   // read again only behind the next round's barrier
    sh.num[tid] = 0;
    if (tid == 0) sh.num[kBinSlots] = 0;
    __syncthreads ();
    n_list = sh.n_next;
    if (n_list == 0) break;
  }
}

} // namespace drx
