// axsq_query.hip -- BVH candidate search (findPoints / findBoundingBoxes / findRays).
//
// Reference: LinearBVH::findCandidatesImpl (src/axom/spin/policy/LinearBVH.hpp:273-402),
// GPU form: count pass, exclusive scan, fill pass (:296-367). One lane per
// query; candidates of query i are written in traversal order at offsets[i],
// at most counts[i] of them (the fill raises kStatusFillMismatch in the status word
// when its walk finds another number, so a caller whose inputs changed after
// the count gets an error and no write past its buffer). In the one-call
// search the count pass also keeps each query's first kstash candidate ids and
// lists the queries that have more, so the fill copies the kept ids and
// searches again only for the listed queries.
//
// Points and boxes walk the compact nodes of axsq_find.hpp in either traversal
// form (k_find_compact), rays too, a wave for several rays (k_ray_count) or for
// one (k_ray_fill). Trees whose coordinates are out of those nodes' range or below
// their resolution, and searches whose visits are counted, walk the FP64 nodes, a
// lane per query on the vote schedule (k_find). A query's nodes are met left
// before right in all of them, so lists and order are the same.
#include "axsq_internal.hpp"
#include "axsq_traverse.hpp"

namespace axsq {

namespace {

struct FindArgs {
  const Node64* nodes;
  const FindNode* fnodes;
  FindSpace space;
  const double* leaf_boxes;
  const int32_t* leaf_ids;
  const void* x;  // double queries, or float ones for a float tree (f32)
  const void* y;
  const void* z;
  int64_t stride;
  int f32;  // a float tree: float queries, the ray test in float
  int64_t nq;
  int dims;  // 2: queries are 2-D (z = 0)
  int32_t ninner;
  double tol;
  int32_t* counts;           // count pass: output
  const int32_t* fill_cnt;   // fill: each query's room, the counts its count pass wrote
  const int32_t* offsets;
  int32_t* cands;
  int pairs;  // fill: cands takes (query, id) records
  int32_t* status;
  int32_t* stash;      // count pass: kstash leaf positions per query (or NULL)
  int kstash;
  int32_t* stash_cnt;  // count pass: a copy of the counts
  int32_t* over;       // count pass: queries with more than kstash; fill: those to search
  uint32_t* nover;
  unsigned long long* visits;  // count pass: sum of the walks' inner-node visits (or NULL)
};

enum { kCountPass = 0, kFillAll = 1, kFillListed = 2 };

// Predicates of BVH.hpp:499-501 (contains), :558-560 (intersectsWith),
// :529-532 (intersect_ray with the BVH tolerance).
template <int KIND>
__device__ __forceinline__ bool pred64(const double* prim, const double* inv, double tol,
                                       const double b[6], int f32 = 0, int dims = 3) {
  if (KIND == AXSQ_QUERY_POINTS) {
    return !(prim[0] < b[0] || prim[0] > b[3] || prim[1] < b[1] || prim[1] > b[4] ||
             prim[2] < b[2] || prim[2] > b[5]);
  } else if (KIND == AXSQ_QUERY_BOXES) {
    return (prim[3] >= b[0] && prim[0] <= b[3]) && (prim[4] >= b[1] && prim[1] <= b[4]) &&
           (prim[5] >= b[2] && prim[2] <= b[5]);
  } else {
    return f32 ? ray_box_f32(prim, b, (float)tol, dims) : ray_box(prim, inv, b, tol);
  }
}

// Stack entries per lane in LDS: a point's or box's walk pushes one entry per
// node where both children hold the query, rarely many, so 16 (deeper ones in
// the private array) let 8 waves per SIMD share a CU's LDS instead of 5
// (findPoints 1M x 100k 0.486 -> 0.461 ms; the hex candidate search 0.86 ->
// 0.77 ms). Ray walks keep 32.
template <int KIND>
constexpr int find_lds_stack() { return KIND == AXSQ_QUERY_RAYS ? kLdsStack : 16; }

__device__ __forceinline__ void load_leaf_box(const double* __restrict__ leaf_boxes, int32_t pos,
                                              double lb[6]) {
  const double2* p = reinterpret_cast<const double2*>(leaf_boxes + 6 * (int64_t)pos);
  const double2 c0 = p[0], c1 = p[1], c2 = p[2];
  lb[0] = c0.x; lb[1] = c0.y; lb[2] = c1.x; lb[3] = c1.y; lb[4] = c2.x; lb[5] = c2.y;
}

// Query i in FP64 (2-D: z = 0; a box: min, max; a ray: origin, direction).
template <int KIND>
__device__ __forceinline__ void load_prim(const FindArgs& a, int64_t i, double prim[6]) {
  // element k of query array p (float queries widen exactly)
  auto ld = [&](const void* p, int64_t k) -> double {
    return a.f32 ? (double)static_cast<const float*>(p)[k] : static_cast<const double*>(p)[k];
  };
  if (KIND == AXSQ_QUERY_POINTS) {
    prim[0] = ld(a.x, i * a.stride);
    prim[1] = ld(a.y, i * a.stride);
    prim[2] = (a.dims == 2) ? 0.0 : ld(a.z, i * a.stride);
    prim[3] = prim[4] = prim[5] = 0.0;
  } else if (a.dims == 2) {  // box: min x y, max x y; ray: origin x y, direction x y
    const int64_t o = i * a.stride;
    prim[0] = ld(a.x, o);
    prim[1] = ld(a.x, o + 1);
    prim[2] = 0.0;
    prim[3] = ld(a.x, o + 2);
    prim[4] = ld(a.x, o + 3);
    prim[5] = 0.0;
  } else {
    for (int k = 0; k < 6; ++k) prim[k] = ld(a.x, i * a.stride + k);
  }
}

// Candidate k of the whole search: query i's id.
__device__ __forceinline__ void put_cand(const FindArgs& a, int64_t k, int64_t i, int32_t id) {
  if (a.pairs)
    reinterpret_cast<int2*>(a.cands)[k] = make_int2((int32_t)i, id);
  else
    a.cands[k] = id;
}

// The end of a count pass: lists the queries with more than kstash ids, one
// list slot per wave.
__device__ __forceinline__ void list_over(const FindArgs& a, bool more, int64_t i) {
  const uint64_t m = __ballot(more);
  if (m) {
    const int lane = (int)__lane_id();
    const int leader = __ffsll((unsigned long long)m) - 1;
    uint32_t base = 0;
    if (lane == leader) base = atomicAdd(a.nover, (uint32_t)__popcll(m));
    base = __shfl(base, leader);
    const uint64_t below = (lane == 0) ? 0ull : (m & ((~0ull) >> (64 - lane)));
    if (more) a.over[base + __popcll(below)] = (int32_t)i;
  }
}

template <int KIND, int MODE>
__global__ __launch_bounds__(kBlock) void k_find(FindArgs a) {
  constexpr bool FILL = MODE != kCountPass;
  constexpr int kLds = find_lds_stack<KIND>();
  __shared__ int32_t s_stack[stack_lds_words<kLds>(kBlock)];
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = j < a.nq;
  if (FILL && !live) return;  // the count pass keeps whole waves for its ballot
  int32_t count = 0;
  int64_t i = 0;
  if (live) {
    i = (MODE == kFillListed) ? (int64_t)a.over[j] : j;
    lds_i32* stk = lane_stack_base<kLds>(s_stack);
    double prim[6];
    load_prim<KIND>(a, i, prim);
    const int32_t offset = FILL ? a.offsets[i] : 0;
    const int32_t room = FILL ? a.fill_cnt[i] : 0;
    int32_t* const stash = (!FILL && a.stash) ? a.stash + i * a.kstash : nullptr;
    auto emit = [&](int32_t pos) {
      if (FILL) {
        if (count < room) put_cand(a, (int64_t)offset + count, i, a.leaf_ids[pos]);
      } else {
        if (stash && count < a.kstash) stash[count] = pos;
      }
      ++count;
    };
    auto no_pref = [](const auto*, const auto*) { return false; };
    double inv[3] = {0.0, 0.0, 0.0};
    if (KIND == AXSQ_QUERY_RAYS)
      for (int d = 0; d < 3; ++d) inv[d] = 1.0 / prim[3 + d];
    // the walk tests a child box only when its validity bit is set, so an
    // invalid box (min > max on some axis) is never entered
    const int32_t v = traverse_voted<Node64, double, kLds>(
        a.nodes, a.ninner, stk,
        [&](const double* b) { return pred64<KIND>(prim, inv, a.tol, b, a.f32, a.dims); }, no_pref,
        emit);
    if (v < 0) atomicOr(a.status, kStatusStack);
    if (!FILL && a.visits && v > 0) atomicAdd(a.visits, (unsigned long long)v);
    if (FILL && count != room) atomicOr(a.status, kStatusFillMismatch);
    if (!FILL) {
      a.counts[i] = count;
      if (stash) a.stash_cnt[i] = count;
    }
  }
  if (!FILL && a.stash) list_over(a, live && count > a.kstash, i);
}

// The point and box searches on the compact nodes, one lane per query. A leaf
// is taken where the walk meets it, so the lanes of a wave only visit nodes;
// the kept ids are leaf positions (the copy looks the ids up), so no load
// stands in a visit's way. The ring of pending children is k_sdf_cull's.
// 1M points into 100,000 boxes, 3-D / 2-D (18.9 / 48.5 visits each): 329 / 1,060
// us with the FP64 nodes and the vote schedule, 168 / 532 here.
template <int KIND, int MODE, int DIMS>
__global__ __launch_bounds__(kBlock) void k_find_compact(FindArgs a) {
  constexpr bool FILL = MODE != kCountPass;
  constexpr bool BOX = KIND == AXSQ_QUERY_BOXES;
  constexpr int kRing = 16;
  __shared__ uint32_t s_ring[kRing * kBlock];
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = j < a.nq;
  if (FILL && !live) return;  // the count pass keeps whole waves for its ballot
  int32_t count = 0;
  int64_t i = 0;
  if (live) {
    i = (MODE == kFillListed) ? (int64_t)a.over[j] : j;
    typedef __attribute__((address_space(3))) uint32_t lds_u32;
    lds_u32* ring = (lds_u32*)(s_ring + (threadIdx.x / kWaveLanes) * (kRing * kWaveLanes) +
                               threadIdx.x % kWaveLanes);
    uint32_t deep[kStack];
    double prim[6];
    load_prim<KIND>(a, i, prim);
    FindQuery<BOX> q;
    q.init(a.space, prim);
    const int32_t offset = FILL ? a.offsets[i] : 0;
    const int32_t room = FILL ? a.fill_cnt[i] : 0;
    int32_t* const stash = (!FILL && a.stash) ? a.stash + i * a.kstash : nullptr;
    bool bad = false;
    auto leaf = [&](uint32_t code) {
      const int32_t pos = (int32_t)(code & kFindPos);
      if (!(code & kFindSureBit)) {
        double lb[6];
        load_leaf_box(a.leaf_boxes, pos, lb);
        if (!(valid6(lb) && pred64<KIND>(prim, nullptr, a.tol, lb))) return;
      }
      if (FILL) {
        if (count < room) put_cand(a, (int64_t)offset + count, i, a.leaf_ids[pos]);
      } else {
        if (stash && count < a.kstash) stash[count] = pos;
      }
      ++count;
    };
    uint32_t cur = 0;
    int32_t sp = -1, base = 0, visits = 0;  // entries base .. sp are in the ring, below in deep
    // a box with a NaN coordinate overlaps nothing; a point of NaNs alone is in
    // every valid box, and no distance tells the invalid ones, so never sure
    bool none = true;
    for (int d = 0; d < (BOX ? 6 : DIMS); ++d) {
      const bool nan = __builtin_isnan(prim[d]);
      if (BOX && nan) cur = kFindEnd;
      none = none && nan;
    }
    const float sure = none ? -INFINITY : -kFindSure;
    while (cur != kFindEnd) {
      float gl, gr;
      uint32_t lc, rc;
      find_visit<BOX, DIMS>(a.fnodes, cur, q, gl, gr, lc, rc);
      const bool in_l = !(gl > 0.0f), in_r = !(gr > 0.0f);
      if (!(gl < sure)) lc &= ~(lc & kFindLeaf ? kFindSureBit : 0u);
      if (!(gr < sure)) rc &= ~(rc & kFindLeaf ? kFindSureBit : 0u);
      if (++visits > a.ninner) {  // only a malformed tree
        bad = true;
        break;
      }
      cur = in_l ? lc : in_r ? rc : kFindEnd;
      if (in_l && in_r) {
        ++sp;
        if (sp - base >= kRing) {
          deep[base] = ring[(base & (kRing - 1)) * kWaveLanes];
          ++base;
        }
        if (sp >= kStack) {
          bad = true;
          break;
        }
        ring[(sp & (kRing - 1)) * kWaveLanes] = rc;
      }
      while (cur & kFindLeaf) {  // leaves, and the next pending child
        if (cur != kFindEnd) leaf(cur);
        if (sp < 0) {
          cur = kFindEnd;
          break;
        }
        if (sp < base)
          cur = deep[--base];
        else
          cur = ring[(sp & (kRing - 1)) * kWaveLanes];
        --sp;
      }
    }
    if (bad) atomicOr(a.status, kStatusStack);
    if (FILL && count != room) atomicOr(a.status, kStatusFillMismatch);
    if (!FILL) {
      a.counts[i] = count;
      if (stash) a.stash_cnt[i] = count;
    }
  }
  if (!FILL && a.stash) list_over(a, live && count > a.kstash, i);
}

// One visit for a ray: on the compact node, or, for a ray outside their range
// (ok false), the exact test on the FP64 node.
template <int DIMS>
__device__ __forceinline__ void ray_visit(const FindArgs& a, uint32_t node, const FindRay& q,
                                          bool ok, const double* prim, const double* inv,
                                          bool& in_l, bool& in_r, uint32_t& lc, uint32_t& rc) {
  find_visit_ray<DIMS>(a.fnodes, node, q, in_l, in_r, lc, rc);
  if (!ok) {
    double l[6], r[6];
    int32_t l2, r2, flags;
    load_node(a.nodes, (int32_t)node, l, r, l2, r2, flags);
    in_l = (flags & 1) && pred64<AXSQ_QUERY_RAYS>(prim, inv, a.tol, l, a.f32, a.dims);
    in_r = (flags & 2) && pred64<AXSQ_QUERY_RAYS>(prim, inv, a.tol, r, a.f32, a.dims);
  }
}

__device__ __forceinline__ bool ray_leaf(const FindArgs& a, int32_t pos, const double* prim,
                                         const double* inv) {
  double lb[6];
  load_leaf_box(a.leaf_boxes, pos, lb);
  return valid6(lb) && pred64<AXSQ_QUERY_RAYS>(prim, inv, a.tol, lb, a.f32, a.dims);
}

// The count pass for rays. A ray's walk is long (132 visits among 100,000
// boxes), of very different lengths, and serial, so one lane per ray leaves
// most lanes waiting for the wave's longest walk and the chip for the longest
// of all. Here a wave walks for `rays` rays together (find_pooled). A ray's
// leaves so come in any order; their positions are the walk's order, which
// k_stash_order restores.
// 100,000 rays, 100,000 boxes: 965 us one lane per ray on the FP64 nodes, 662 on
// the compact ones, 129 here.
constexpr int kPoolRays = 32;
template <int DIMS>
__global__ __launch_bounds__(kWaveLanes) void k_ray_count(FindArgs a, int rays) {
  __shared__ FindPool s_pool;
  __shared__ double s_prim[9][kPoolRays];  // origin, direction, 1 / direction
  __shared__ float s_q[3 * DIMS][kPoolRays];
  __shared__ int32_t s_count[kPoolRays], s_ok[kPoolRays];
  const int lane = (int)threadIdx.x;
  const int64_t i = (int64_t)blockIdx.x * rays + lane;
  const bool mine = lane < rays && i < a.nq;
  if (mine) {
    double prim[6];
    load_prim<AXSQ_QUERY_RAYS>(a, i, prim);
    FindRay q;
    s_ok[lane] = q.init(a.space, prim, a.tol, a.f32);
    for (int d = 0; d < 6; ++d) s_prim[d][lane] = prim[d];
    for (int d = 0; d < 3; ++d) s_prim[6 + d][lane] = 1.0 / prim[3 + d];
    for (int d = 0; d < DIMS; ++d) {
      s_q[3 * d][lane] = q.h[d];
      s_q[3 * d + 1][lane] = q.l[d];
      s_q[3 * d + 2][lane] = q.inv[d];
    }
    s_count[lane] = 0;
  }
  const bool done = find_pooled(
      s_pool, mine, a.ninner,
      [&](uint32_t node, int who, bool& in_l, bool& in_r, uint32_t& lc, uint32_t& rc) {
        FindRay q;
        for (int d = 0; d < DIMS; ++d) {
          q.h[d] = s_q[3 * d][who];
          q.l[d] = s_q[3 * d + 1][who];
          q.inv[d] = s_q[3 * d + 2][who];
        }
        const bool ok = s_ok[who];
        double prim[6], inv[3];
        if (!ok) {
          for (int d = 0; d < 6; ++d) prim[d] = s_prim[d][who];
          for (int d = 0; d < 3; ++d) inv[d] = s_prim[6 + d][who];
        }
        ray_visit<DIMS>(a, node, q, ok, prim, inv, in_l, in_r, lc, rc);
      },
      [&](int32_t pos, int who) {
        double prim[6], inv[3];
        for (int d = 0; d < 6; ++d) prim[d] = s_prim[d][who];
        for (int d = 0; d < 3; ++d) inv[d] = s_prim[6 + d][who];
        if (!ray_leaf(a, pos, prim, inv)) return;
        const int32_t c = atomicAdd(&s_count[who], 1);
        if (a.stash && c < a.kstash)
          a.stash[((int64_t)blockIdx.x * rays + who) * a.kstash + c] = pos;
      });
  if (!done && lane == 0) atomicOr(a.status, kStatusStack);
  wave_sync();
  const int32_t c = mine ? s_count[lane] : 0;
  if (mine) {
    a.counts[i] = c;
    if (a.stash) a.stash_cnt[i] = c;
  }
  if (a.stash) list_over(a, mine && c > a.kstash, i);
}

// The fill pass for rays: a wave per ray (find_ordered).
// 20,000 boxes in the plane, 50,000 rays of 134 candidates, the whole search:
// 3,790 us with a lane per ray on the FP64 nodes, 500 here.
template <int MODE, int DIMS>
__global__ __launch_bounds__(kWaveLanes) void k_ray_fill(FindArgs a) {
  __shared__ uint32_t s_item[kOrderedItems];
  const int lane = (int)threadIdx.x;
  for (int64_t j = blockIdx.x; j < a.nq; j += gridDim.x) {
    const int64_t i = (MODE == kFillListed) ? (int64_t)a.over[j] : j;
    double prim[6], inv[3];
    load_prim<AXSQ_QUERY_RAYS>(a, i, prim);
    for (int d = 0; d < 3; ++d) inv[d] = 1.0 / prim[3 + d];
    FindRay q;
    const bool ok = q.init(a.space, prim, a.tol, a.f32);
    const int32_t offset = a.offsets[i], room = a.fill_cnt[i];
    const int32_t count = find_ordered(
        s_item, a.ninner,
        [&](uint32_t node, bool& in_l, bool& in_r, uint32_t& lc, uint32_t& rc) {
          ray_visit<DIMS>(a, node, q, ok, prim, inv, in_l, in_r, lc, rc);
        },
        [&](int32_t pos) { return ray_leaf(a, pos, prim, inv); },
        [&](int32_t c, int32_t pos) {
          if (c < room) a.cands[offset + c] = a.leaf_ids[pos];
        });
    if (lane == 0 && count < 0) atomicOr(a.status, kStatusStack);
    if (lane == 0 && count != room) atomicOr(a.status, kStatusFillMismatch);
  }
}

// The fill pass for queries with at most kstash (<= 64) candidates: the ids of
// the leaf positions the count pass kept, at offsets[i]. What a wave's 64
// queries kept is taken as one run, 64 ids at a time, each lane finding its
// query among the 64 places in the run; four such steps' loads are in flight at
// once. Queries with more ids have no place in it, however many those are. Where
// no query has more than 4 ids a lane copies its own.
// 1M queries of 12 ids: 84 us with a query at a time over the wave, 48 here.
template <bool PAIRS>
__global__ __launch_bounds__(kBlock) void k_stash_copy(const int32_t* __restrict__ stash,
                                                        int kstash,
                                                        const int32_t* __restrict__ stash_cnt,
                                                        const int32_t* __restrict__ offsets,
                                                        const int32_t* __restrict__ leaf_ids,
                                                        int64_t nq, int32_t* __restrict__ cands) {
  __shared__ int32_t s_at[kBlock], s_off[kBlock];
  const int lane = (int)__lane_id();
  int32_t* at = s_at + (threadIdx.x - lane);    // a query's place in the run
  int32_t* off = s_off + (threadIdx.x - lane);  // and in the output
  const int64_t base = (int64_t)blockIdx.x * blockDim.x + threadIdx.x - lane;  // the wave's first
  if (base >= nq) return;  // the whole wave
  auto put = [&](int32_t k, int64_t i, int32_t id) {
    if (PAIRS)
      reinterpret_cast<int2*>(cands)[k] = make_int2((int32_t)i, id);
    else
      cands[k] = id;
  };
  const int64_t mine = base + lane;
  int32_t c = (mine < nq) ? stash_cnt[mine] : 0;
  const int32_t o = (mine < nq) ? offsets[mine] : 0;
  if (c > kstash) c = 0;  // listed: searched again
  if (__ballot(c > 4) == 0) {  // few ids everywhere
    for (int32_t k = 0; k < c; ++k) put(o + k, mine, leaf_ids[stash[mine * kstash + k]]);
    return;
  }
  int32_t end = c;  // of this lane's part of the run, at most 64 * 64
  for (int step = 1; step < kWaveLanes; step <<= 1) {
    const int32_t v = __shfl_up(end, step);
    if (lane >= step) end += v;
  }
  at[lane] = end - c;
  off[lane] = o;
  wave_sync();
  const int32_t run = __shfl(end, kWaveLanes - 1);
  for (int32_t j0 = lane; j0 - lane < run; j0 += 4 * kWaveLanes) {
    int32_t id[4], to[4];
    int q[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int32_t j = j0 + u * kWaveLanes;
      q[u] = 0;  // the last query whose part starts at or before j
#pragma unroll
      for (int step = kWaveLanes / 2; step > 0; step >>= 1)
        if (at[q[u] + step] <= j) q[u] += step;
      const int32_t k = j - at[q[u]];
      to[u] = j < run ? off[q[u]] + k : 0;
      id[u] = j < run ? stash[(base + q[u]) * kstash + k] : 0;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (j0 + u * kWaveLanes < run) id[u] = leaf_ids[id[u]];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (j0 + u * kWaveLanes < run) put(to[u], base + q[u], id[u]);
  }
}

// The same for rays, whose positions were kept in any order: in order of
// position. A wave takes 16 rays, one after the other, lane l placing id l by
// the number of smaller ones (100,000 rays: 55 us with 64 rays a wave, 23 with 16).
constexpr int kCopyRays = 16;
__global__ __launch_bounds__(kBlock) void k_stash_order(const int32_t* __restrict__ stash,
                                                         int kstash,
                                                         const int32_t* __restrict__ stash_cnt,
                                                         const int32_t* __restrict__ offsets,
                                                         const int32_t* __restrict__ leaf_ids,
                                                         int64_t nq, int32_t* __restrict__ cands) {
  const int lane = (int)__lane_id();
  const int64_t base =
      ((int64_t)blockIdx.x * blockDim.x + threadIdx.x - lane) / kWaveLanes * kCopyRays;
  if (base >= nq) return;  // the whole wave
  const int64_t mine = base + lane;
  const bool has = lane < kCopyRays && mine < nq;
  const int32_t c_me = has ? stash_cnt[mine] : 0;
  const int32_t o_me = has ? offsets[mine] : 0;
  for (int j0 = 0; j0 < kCopyRays; j0 += 8) {
    int32_t v[8], cc[8], oo[8], at[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      cc[u] = __shfl(c_me, j0 + u);
      oo[u] = __shfl(o_me, j0 + u);
      const bool take = cc[u] <= kstash && lane < cc[u];
      v[u] = take ? stash[(base + j0 + u) * kstash + lane] : 0;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int c = cc[u] <= kstash ? __builtin_amdgcn_readfirstlane(cc[u]) : 0;
      at[u] = 0;
      for (int t = 0; t < c; ++t) at[u] += __builtin_amdgcn_readlane(v[u], t) < v[u];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (cc[u] <= kstash && lane < cc[u]) v[u] = leaf_ids[v[u]];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (cc[u] <= kstash && lane < cc[u]) cands[oo[u] + at[u]] = v[u];
  }
}

template <int MODE>
hipError_t launch_mode(int kind, bool compact, const FindArgs& a, hipStream_t s) {
  const unsigned g = grid_for(a.nq);
  if (kind == AXSQ_QUERY_RAYS) {
    if (!compact) {
      k_find<AXSQ_QUERY_RAYS, MODE><<<g, kBlock, 0, s>>>(a);
    } else if constexpr (MODE == kCountPass) {
      // few rays: fewer a wave, to fill the chip's 5,120 waves of this kernel
      // (10,000 rays at 2 / 8 / 32 a wave: 191 / 201 / 262 us; 100,000 at 8 / 16 /
      // 32: 289 / 299 / 284)
      int rays = 1;
      while (rays < kPoolRays && a.nq > (int64_t)rays * 5120) rays *= 2;
      const unsigned gr = (unsigned)((a.nq + rays - 1) / rays);
      if (a.dims == 2)
        k_ray_count<2><<<gr, kWaveLanes, 0, s>>>(a, rays);
      else
        k_ray_count<3><<<gr, kWaveLanes, 0, s>>>(a, rays);
    } else {
      const unsigned gr = (unsigned)std::min<int64_t>(a.nq, int64_t(1) << 20);
      if (a.dims == 2)
        k_ray_fill<MODE, 2><<<gr, kWaveLanes, 0, s>>>(a);
      else
        k_ray_fill<MODE, 3><<<gr, kWaveLanes, 0, s>>>(a);
    }
  } else if (kind == AXSQ_QUERY_POINTS) {
    if (!compact)
      k_find<AXSQ_QUERY_POINTS, MODE><<<g, kBlock, 0, s>>>(a);
    else if (a.dims == 2)
      k_find_compact<AXSQ_QUERY_POINTS, MODE, 2><<<g, kBlock, 0, s>>>(a);
    else
      k_find_compact<AXSQ_QUERY_POINTS, MODE, 3><<<g, kBlock, 0, s>>>(a);
  } else {
    if (!compact)
      k_find<AXSQ_QUERY_BOXES, MODE><<<g, kBlock, 0, s>>>(a);
    else if (a.dims == 2)
      k_find_compact<AXSQ_QUERY_BOXES, MODE, 2><<<g, kBlock, 0, s>>>(a);
    else
      k_find_compact<AXSQ_QUERY_BOXES, MODE, 3><<<g, kBlock, 0, s>>>(a);
  }
  return hipGetLastError();
}

}  // namespace

// mode 0: count (and keep the first kstash leaf positions when stash is given);
// 1: fill every query; 2: fill the nq queries listed in `over`.
int find_launch(const axsq_bvh* b, int kind, int mode, const void* x, const void* y,
                const void* z, int64_t stride, int64_t nq, double tol, int32_t* counts,
                const int32_t* fill_cnt, const int32_t* offsets, int32_t* cands, int32_t* stash,
                int kstash, int32_t* stash_cnt, int32_t* over, uint32_t* nover, hipStream_t s,
                bool pairs) {
  FindArgs a;
  a.nodes = b->nodes;
  a.fnodes = b->fnodes;
  a.leaf_boxes = b->leaf_boxes;
  a.leaf_ids = b->leaf_ids;
  a.x = x;
  a.y = y;
  a.z = z;
  a.stride = stride;
  a.f32 = b->f32 ? 1 : 0;
  a.nq = nq;
  a.dims = b->dims;
  a.ninner = (int32_t)(b->n - 1);
  a.tol = tol;
  a.counts = counts;
  a.fill_cnt = fill_cnt;
  a.offsets = offsets;
  a.cands = cands;
  a.pairs = pairs;
  a.status = b->status;
  a.stash = stash;
  a.kstash = kstash;
  a.stash_cnt = stash_cnt;
  a.over = over;
  a.nover = nover;
  a.visits = (mode == kCountPass && b->stats) ? b->find_visits : nullptr;
  // with visits counted, the FP64 nodes: the count is the reference traversal's
  const bool compact = b->find_ok && !a.visits && find_space(b->bounds, a.space);
  ProfRange pr(mode == kCountPass ? "bvh_find_count" : "bvh_find_fill", s);
  const hipError_t e = mode == kCountPass ? launch_mode<kCountPass>(kind, compact, a, s)
                       : mode == kFillAll ? launch_mode<kFillAll>(kind, compact, a, s)
                                          : launch_mode<kFillListed>(kind, compact, a, s);
  pr.stop();
  if (e != hipSuccess) {
    set_error("find kernel launch failed: %s", hipGetErrorString(e));
    return AXSQ_ERR_HIP;
  }
  return AXSQ_OK;
}

int stash_copy_launch(const axsq_bvh* b, int kind, bool pairs, const int32_t* stash, int kstash,
                      const int32_t* stash_cnt, const int32_t* offsets, int64_t nq,
                      int32_t* cands, hipStream_t s) {
  if (nq <= 0) return AXSQ_OK;
  ProfRange pr("bvh_find_copy", s);
  if (kind == AXSQ_QUERY_RAYS && b->find_ok) {
    k_stash_order<<<grid_for((nq + kCopyRays - 1) / kCopyRays * kWaveLanes), kBlock, 0, s>>>(
        stash, kstash, stash_cnt, offsets, b->leaf_ids, nq, cands);
  } else {
    auto* const copy = pairs ? k_stash_copy<true> : k_stash_copy<false>;
    copy<<<grid_for(nq), kBlock, 0, s>>>(stash, kstash, stash_cnt, offsets, b->leaf_ids, nq,
                                         cands);
  }
  AXSQ_CHECK_HIP(hipGetLastError());
  return AXSQ_OK;
}

}  // namespace axsq
