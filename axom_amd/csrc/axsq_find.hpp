// axsq_find.hpp -- compact nodes for the searches.
//
// Those searches are bound by the bytes a visit reads: the lanes of a wave are
// at different nodes, the vector L1 returns 16 bytes of one lane a cycle, and
// a visit of the 128-byte FP64 node takes seven such reads (its FP32 form
// four). This node takes three (two in 2-D): both child boxes as halves, rounded outward,
// relative to a float centre and scaled to the node's own size.
//
// Exactness. A candidate is a leaf whose FP64 box passes the FP64 test: a box
// contains its children's boxes bit for bit, so a leaf that passes is reached
// whatever its ancestors' tests. The walk here reaches every leaf whose
// outward box passes, in the same order (left before right), and takes it at
// once where the query is inside by more than all rounding could give
// (kFindSure of the node's size), and after the FP64 test otherwise. So ids,
// counts and order are those of the FP64 walk.
//
// Rounding. Query coordinates are taken relative to the root box's centre,
// times a power of two (FindSpace), and split into two floats; a node's t is
// their difference to its centre, times its scale s, in two fused steps, so
// that it is off by at most 2^-22 near the box's faces, and by s 2^-46 from
// the split. The build widens the extents by 2^-20 + s 2^-44. Boxes down to
// about 2^-36 of the root box keep their own resolution.
#pragma once

#include <hip/hip_fp16.h>
#include <math.h>

#include "axsq_device.hpp"

namespace axsq {

// Coordinates of the searches: (x - o) * scale, the root box's longest side
// between 1 and 2. ok: finite, in range and not a point, from which no size of
// the tree could be told (100,000 equal boxes without extent, 10,000 points
// elsewhere: every node visited, 75 ms; 0.07 with the FP64 nodes); else the FP64
// nodes are walked.
struct FindSpace {
  double o[3];
  double scale;
};

__host__ __device__ inline bool find_space(const double b[6], FindSpace& fs) {
  double ext = 0.0;
  bool ok = true;
  for (int d = 0; d < 3; ++d) {
    const double e = b[3 + d] - b[d];
    ok = ok && b[d] >= -1e100 && b[3 + d] <= 1e100 && e >= 0.0;
    if (e > ext) ext = e;
    fs.o[d] = 0.5 * (b[d] + b[3 + d]);
  }
  int e2 = 0;
  (void)frexp(ext, &e2);
  ok = ok && ext > 0.0 && e2 > -330;
  fs.scale = ldexp(1.0, 1 - (e2 > -330 ? e2 : -330));
  return ok;
}

// Child boxes along x, y, z: l[d] / r[d] are halves lo | hi << 16 of
// (X - c) * s, X in the search's coordinates, cs = -c * s. Links: an inner
// node's index, or a leaf position with bit 31 and, where the node's scale
// lets a test be sure, bit 30 set.
struct __attribute__((aligned(16))) FindNode {
  float cs[3];
  float s;
  uint32_t l[3], r[3];
  uint32_t lc, rc;
};
static_assert(sizeof(FindNode) == 48, "FindNode is three 16-byte loads");

// A 2-D tree's node, two loads: no z, and the scale in the lowest three bits of
// the two centres (whose own values have them zero). 100,000 nodes take 3.2 MB
// and stay in one XCD's L2, where 48 bytes each did not. 1M points into 100,000
// boxes in the plane: 640 us with 48 bytes, 532 with 32.
struct __attribute__((aligned(16))) FindNode2 {
  uint32_t cs[2];
  uint32_t l[2], r[2];
  uint32_t lc, rc;
};
static_assert(sizeof(FindNode2) == 32, "FindNode2 is two 16-byte loads");

constexpr uint32_t kFindLeaf = 0x80000000u, kFindSureBit = 0x40000000u;
constexpr uint32_t kFindPos = 0x3fffffffu;
constexpr uint32_t kFindEnd = kFindLeaf | kFindPos;  // no leaf has that position
constexpr uint32_t kFindNone = 0xfc007c00u;  // an invalid child's range, from +inf to -inf
// Inside by this much of the node's scale is inside the FP64 box: extents are
// below 2, but with their margins may round out past it, so the halves are off
// by 2^-9 at most; the margins of a node with the bit set (s up to 2^30) and the
// query's t by less than 2^-13 together.
constexpr float kFindSure = 0.00219726562f;  // 2^-9 + 2^-12
constexpr float kFindFar = 3e38f;  // beyond every far end of a ray's interval

// Halves rounded outward (sign and magnitude, so the next one down or up is
// one off in its bits).
__device__ __forceinline__ uint32_t half_range(float lo, float hi) {
  uint16_t l = __half_as_ushort(__float2half_rn(lo)), h = __half_as_ushort(__float2half_rn(hi));
  if (__half2float(__ushort_as_half(l)) > lo)
    l = (l & 0x8000u) ? l + 1 : (l == 0 ? 0x8001u : l - 1);
  if (__half2float(__ushort_as_half(h)) < hi)
    h = (h & 0x8000u) ? (h == 0x8000u ? 1 : h - 1) : h + 1;
  return (uint32_t)l | ((uint32_t)h << 16);
}

// lo - t and t - hi with the halves taken as they are (v_fma_mix_f32: one
// instruction, no conversion).
__device__ __forceinline__ float half_lo_minus(uint32_t ext, float t) {
  float r;
  asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(ext), "v"(t));
  return r;
}
__device__ __forceinline__ float half_minus_hi(uint32_t ext, float t) {
  float r;
  asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
      : "=v"(r)
      : "v"(ext), "v"(t));
  return r;
}

// The node of children l, r (valid by `flags` bits 0 and 1) with links lc, rc
// (inner index or -(leaf + 1)). dims 2: the z range never decides.
__device__ __forceinline__ FindNode make_find_node(const FindSpace& fs, int dims,
                                                   const double l[6], const double r[6],
                                                   int32_t flags, int32_t lc, int32_t rc) {
  FindNode n;
  float c[3];
  double X[2][6], m = 0.0;
  for (int d = 0; d < 6; ++d) {
    X[0][d] = (l[d] - fs.o[d % 3]) * fs.scale;
    X[1][d] = (r[d] - fs.o[d % 3]) * fs.scale;
  }
  for (int d = 0; d < 3; ++d) {
    const double lo = (flags & 1) ? ((flags & 2) ? fmin(X[0][d], X[1][d]) : X[0][d]) : X[1][d];
    const double hi = (flags & 1) ? ((flags & 2) ? fmax(X[0][3 + d], X[1][3 + d]) : X[0][3 + d])
                                  : X[1][3 + d];
    c[d] = (flags & 3) ? (float)(0.5 * (lo + hi)) : 0.0f;
    if (dims == 2) c[d] = __uint_as_float(__float_as_uint(c[d]) & ~7u);
    if ((flags & 3) && d < dims) m = fmax(m, fmax(fabs(lo - c[d]), fabs(hi - c[d])));
  }
  // extents below 2; a smaller node, down to a point, spans its margin of at
  // most 2^15, which a half holds
  int e2 = -58;
  if (m > 0.0) (void)frexp(m, &e2);
  e2 = e2 < -58 ? -58 : e2 > 3 ? 3 : e2;
  const double s = ldexp(1.0, 1 - e2);
  const double margin = 9.5367431640625e-07 + s * 5.684341886080802e-14;  // 2^-20 + s 2^-44
  n.s = (float)s;
  for (int d = 0; d < 3; ++d) {
    n.cs[d] = (float)(-(double)c[d] * s);
    for (int k = 0; k < 2; ++k) {
      uint32_t e = kFindNone;
      if (flags & (1 << k)) {
        const double lo = d < dims ? (X[k][d] - (double)c[d]) * s - margin : -2.0;
        const double hi = d < dims ? (X[k][3 + d] - (double)c[d]) * s + margin : 2.0;
        e = half_range((float)(lo - fabs(lo) * 1e-7), (float)(hi + fabs(hi) * 1e-7));
      }
      if (k == 0)
        n.l[d] = e;
      else
        n.r[d] = e;
    }
  }
  const uint32_t sure = s <= 1073741824.0 ? kFindSureBit : 0u;  // 2^30
  n.lc = lc >= 0 ? (uint32_t)lc : (kFindLeaf | sure | (uint32_t)(-lc - 1));
  n.rc = rc >= 0 ? (uint32_t)rc : (kFindLeaf | sure | (uint32_t)(-rc - 1));
  return n;
}

// Node i of a tree (dims 2: FindNode2, in the same array).
__device__ __forceinline__ void store_find_node(FindNode* __restrict__ nodes, int32_t i, int dims,
                                                const FindNode& n) {
  if (dims != 2) {
    nodes[i] = n;
    return;
  }
  const uint32_t code = (__float_as_uint(n.s) >> 23) - 125u;  // s = 2^-2 .. 2^59: 0 .. 61
  FindNode2 m;
  m.cs[0] = (__float_as_uint(n.cs[0]) & ~7u) | (code >> 3);
  m.cs[1] = (__float_as_uint(n.cs[1]) & ~7u) | (code & 7u);
  for (int d = 0; d < 2; ++d) {
    m.l[d] = n.l[d];
    m.r[d] = n.r[d];
  }
  m.lc = n.lc;
  m.rc = n.rc;
  reinterpret_cast<FindNode2*>(nodes)[i] = m;
}

// Node i in registers: centres times scale, scale, the children's ranges, links.
template <int DIMS>
__device__ __forceinline__ void load_find_node(const FindNode* __restrict__ nodes, uint32_t i,
                                               float cs[DIMS], float& s, uint32_t el[DIMS],
                                               uint32_t er[DIMS], uint32_t& lc, uint32_t& rc) {
  if constexpr (DIMS == 2) {
    const uint4* p = reinterpret_cast<const uint4*>(reinterpret_cast<const FindNode2*>(nodes) + i);
    const uint4 a = p[0], b = p[1];
    cs[0] = __uint_as_float(a.x & ~7u);
    cs[1] = __uint_as_float(a.y & ~7u);
    s = __uint_as_float(((((a.x & 7u) << 3) | (a.y & 7u)) + 125u) << 23);
    el[0] = a.z;
    el[1] = a.w;
    er[0] = b.x;
    er[1] = b.y;
    lc = b.z;
    rc = b.w;
  } else {
    const float4* p = reinterpret_cast<const float4*>(nodes + i);
    const float4 f = p[0];
    const uint4 a = reinterpret_cast<const uint4*>(p)[1], b = reinterpret_cast<const uint4*>(p)[2];
    cs[0] = f.x;
    cs[1] = f.y;
    cs[2] = f.z;
    s = f.w;
    el[0] = a.x;
    el[1] = a.y;
    el[2] = a.z;
    er[0] = a.w;
    er[1] = b.x;
    er[2] = b.y;
    lc = b.z;
    rc = b.w;
  }
}

// A query's two corners in the search's coordinates, as float pairs (a
// point's are equal). Far coordinates are clamped: outside every box either
// way, and finite times every node's scale (an infinite t less the infinite
// range of an invalid child would be a NaN, which the maximum drops).
template <bool BOX>
struct FindQuery {
  float lh[3], ll[3], hh[BOX ? 3 : 1], hl[BOX ? 3 : 1];
  __device__ __forceinline__ static void split(double x, float& h, float& l) {
    x = x > 1e18 ? 1e18 : x < -1e18 ? -1e18 : x;  // a NaN stays
    h = (float)x;
    l = (float)(x - (double)h);
  }
  __device__ __forceinline__ void init(const FindSpace& fs, const double* prim) {
    for (int d = 0; d < 3; ++d) {
      split((prim[d] - fs.o[d]) * fs.scale, lh[d], ll[d]);
      if constexpr (BOX) split((prim[3 + d] - fs.o[d]) * fs.scale, hh[d], hl[d]);
    }
  }
};

// A visit: the largest signed distance of the query beyond a face of each
// child box, in the node's scale (positive: outside). A point's NaN
// coordinate drops out of the maximum: contains() passes it.
template <bool BOX, int DIMS>
__device__ __forceinline__ void find_visit(const FindNode* __restrict__ nodes, uint32_t cur,
                                           const FindQuery<BOX>& q, float& gl, float& gr,
                                           uint32_t& lc, uint32_t& rc) {
  float cs[DIMS], s;
  uint32_t el[DIMS], er[DIMS];
  load_find_node<DIMS>(nodes, cur, cs, s, el, er, lc, rc);
  gl = gr = -INFINITY;
#pragma unroll
  for (int d = 0; d < DIMS; ++d) {
    const float tl = fmaf(q.ll[d], s, fmaf(q.lh[d], s, cs[d]));
    const float th = BOX ? fmaf(q.hl[d], s, fmaf(q.hh[d], s, cs[d])) : tl;
    gl = fmaxf(fmaxf(half_lo_minus(el[d], th), half_minus_hi(el[d], tl)), gl);
    gr = fmaxf(fmaxf(half_lo_minus(er[d], th), half_minus_hi(er[d], tl)), gr);
  }
}

// Orders a wave's LDS accesses among its lanes (blocks of one wave).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ int lanes_below(uint64_t m) {
  return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                        __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// A ray on the compact nodes. The slab test (FP64, or float in a float tree) of
// a box inside a node's outward box passes only if this one does: in the node's
// coordinates, with the direction over its largest component, each axis gives
// the interval (lo - t) inv .. (hi - t) inv, widened by 2^-20 (|t| + 2) |inv|, at
// least twice its rounding and the exact test's together; the intervals must
// meet at or beyond the origin. An axis whose direction the reference takes as
// zero (inv = 0 here) only tests lo <= t <= hi. The widening also covers a far
// origin's split (2^-48 of it). init returns false for a ray outside the range
// in which neither test overflows or underflows (t up to 2^80, inv to 2^40).
struct FindRay {
  float h[3], l[3];  // the origin as float pairs
  float inv[3];      // largest |direction| / direction; 0: taken as zero
  __device__ __forceinline__ bool init(const FindSpace& fs, const double* ray, double tol,
                                       bool f32) {
    const double m = fmax(fmax(fabs(ray[3]), fabs(ray[4])), fabs(ray[5]));
    const double big = f32 ? 1e15 : 1e100;
    bool ok = !f32 || (fs.scale <= 1e15 && fs.scale >= 1e-15);
    for (int d = 0; d < 3; ++d) {
      const double x = (ray[d] - fs.o[d]) * fs.scale, n = fabs(ray[3 + d]);
      FindQuery<false>::split(x, h[d], l[d]);
      const bool flat = f32 ? fabsf((float)ray[3 + d]) <= (float)tol : near_eq(ray[3 + d], 0.0, tol);
      inv[d] = flat ? 0.0f : (float)(m / ray[3 + d]);
      ok = ok && fabs(x) <= 1048576.0 && fabs(ray[d]) <= big && fabs(fs.o[d]) <= big && n <= big &&
           (flat || (n * big >= 1.0 && m <= n * 1.099511627776e12));
    }
    return ok;
  }
};

template <int DIMS>
__device__ __forceinline__ void find_visit_ray(const FindNode* __restrict__ nodes, uint32_t cur,
                                               const FindRay& q, bool& in_l, bool& in_r,
                                               uint32_t& lc, uint32_t& rc) {
  float cs[DIMS], s;
  uint32_t el[DIMS], er[DIMS];
  load_find_node<DIMS>(nodes, cur, cs, s, el, er, lc, rc);
  float nl = 0.0f, nr = 0.0f, fl = INFINITY, fr = INFINITY;  // near and far ends
#pragma unroll
  for (int d = 0; d < DIMS; ++d) {
    const bool flat = q.inv[d] == 0.0f;
    const float ia = flat ? 1.0f : q.inv[d], ib = flat ? -1.0f : q.inv[d];
    const float t = fmaf(q.l[d], s, fmaf(q.h[d], s, cs[d]));
    const float e = fmaf(fabsf(t), 9.5367432e-7f, 1.9073487e-6f) * fabsf(ia);
    const float a = half_lo_minus(el[d], t) * ia, b = -(half_minus_hi(el[d], t) * ib);
    const float c = half_lo_minus(er[d], t) * ia, g = -(half_minus_hi(er[d], t) * ib);
    // flat: a, b are the distances outside, and only their sign counts
    nl = fmaxf(nl, flat ? (fmaxf(a, b) > e ? INFINITY : 0.0f) : fminf(a, b) - e);
    nr = fmaxf(nr, flat ? (fmaxf(c, g) > e ? INFINITY : 0.0f) : fminf(c, g) - e);
    fl = fminf(fl, flat ? kFindFar : fmaxf(a, b) + e);
    fr = fminf(fr, flat ? kFindFar : fmaxf(c, g) + e);
  }
  in_l = !(nl > fl) && el[0] != kFindNone;
  in_r = !(nr > fr) && er[0] != kFindNone;
}

// Several queries' walks by one wave, in any order: a list of (query, node)
// entries still to visit, of which each step's 64 lanes take the last 64,
// whatever their queries, and a list of reached leaves, taken 64 at a time.
// visit(node, query, in_l, in_r, lc, rc) and leaf(leaf position, query). The
// list cannot overflow: a step takes at most as many entries as leave kFree
// free, each adds at most one net, and near the end one entry at a time walks
// depth first, which a tree of kStack levels fits. False: a malformed tree.
struct FindPool {
  static constexpr int kItems = 512, kLeaves = 192, kFree = kStack;
  uint32_t node[kItems], leaf[kLeaves];
  uint8_t who[kItems], leaf_who[kLeaves];
};

// `mine`: this lane's query takes part (query = lane).
template <class Visit, class Leaf>
__device__ __forceinline__ bool find_pooled(FindPool& l, bool mine, int32_t ninner, Visit&& visit,
                                            Leaf&& take) {
  const int lane = (int)__lane_id();
  const uint64_t has = __ballot(mine);
  if (mine) {
    l.node[lanes_below(has)] = 0;
    l.who[lanes_below(has)] = (uint8_t)lane;
  }
  int n = __popcll(has), nl = 0;  // entries, leaves
  const int64_t limit = (int64_t)n * ninner;
  int64_t visits = 0;
  wave_sync();
  for (;;) {
    if (nl >= kWaveLanes || (n == 0 && nl > 0)) {
      const int m = nl < kWaveLanes ? nl : kWaveLanes;
      nl -= m;
      if (lane < m) take((int32_t)(l.leaf[nl + lane] & kFindPos), (int)l.leaf_who[nl + lane]);
      wave_sync();
      continue;
    }
    if (n == 0) return true;
    const int k = min(min(n, kWaveLanes), max(FindPool::kItems - FindPool::kFree - n, 1));
    visits += k;
    if (visits > limit || n >= FindPool::kItems) return false;
    n -= k;
    bool in_l = false, in_r = false;
    uint32_t lc = 0, rc = 0;
    int who = 0;
    if (lane < k) {
      who = l.who[n + lane];
      visit(l.node[n + lane], who, in_l, in_r, lc, rc);
    }
    wave_sync();  // the entries are read before their places are written
    auto put = [&](bool in, uint32_t code, bool leaves) {
      const bool t = in && ((code & kFindLeaf) != 0) == leaves;
      const uint64_t m = __ballot(t);
      if (leaves) {
        if (t) {
          l.leaf[nl + lanes_below(m)] = code;
          l.leaf_who[nl + lanes_below(m)] = (uint8_t)who;
        }
        nl += __popcll(m);
      } else {
        if (t) {
          l.node[n + lanes_below(m)] = code;
          l.who[n + lanes_below(m)] = (uint8_t)who;
        }
        n += __popcll(m);
      }
    };
    put(in_r, rc, false);
    put(in_l, lc, false);
    put(in_r, rc, true);
    put(in_l, lc, true);
    wave_sync();
  }
}

// One query's walk by a wave, in the walk's order: the pending nodes and
// leaves as a list, the leftmost last; each step takes the last 64, puts each
// node's reached children in its place and hands out the leaves that no node is
// left of. test(leaf position) is asked of those, hit(rank, leaf position)
// called for the ones that pass; returns their number, -1 for a malformed
// tree. The list is bounded as above.
constexpr int kOrderedItems = 512;
template <class Visit, class Test, class Hit>
__device__ __forceinline__ int32_t find_ordered(uint32_t* items, int32_t ninner, Visit&& visit,
                                                Test&& test, Hit&& hit) {
  const int lane = (int)__lane_id();
  int32_t count = 0, visits = 0;
  int n = 1;
  wave_sync();
  if (lane == 0) items[0] = 0;
  wave_sync();
  while (n > 0) {
    const int k = min(min(n, kWaveLanes), max(kOrderedItems - kStack - n, 1));
    const uint32_t item = lane < k ? items[n - 1 - lane] : 0u;
    const bool node = lane < k && !(item & kFindLeaf);
    const uint64_t nodes = __ballot(node);
    const int lead = nodes ? __ffsll((unsigned long long)nodes) - 1 : k;  // leading leaves
    if (lead > 0) {
      const int32_t pos = (int32_t)(item & kFindPos);
      const bool pass = lane < lead && test(pos);
      const uint64_t m = __ballot(pass);
      if (pass) hit(count + lanes_below(m), pos);
      count += __popcll(m);
    }
    visits += __popcll(nodes);
    if (visits > ninner || n >= kOrderedItems) return -1;
    uint32_t first = item, second = item;
    bool one = lane >= lead && lane < k, two = false;
    if (node) {
      bool in_l, in_r;
      uint32_t lc, rc;
      visit(item, in_l, in_r, lc, rc);
      first = in_l ? lc : rc;
      second = rc;
      one = in_l || in_r;
      two = in_l && in_r;
    }
    const uint64_t m1 = __ballot(one), m2 = __ballot(two);
    n += __popcll(m1) + __popcll(m2) - k;
    const int at = n - 1 - lanes_below(m1) - lanes_below(m2);
    wave_sync();  // the entries are read before their places are written
    if (one) items[at] = first;
    if (two) items[at - 1] = second;
    wave_sync();
  }
  return count;
}

}  // namespace axsq
