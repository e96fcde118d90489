// axsq_cull.hip -- builds the oriented child boxes of axsq_cull.hpp over a
// built tree: per leaf its normal (prefix sums, so that a node's mean normal
// is a difference) and closest-point tolerance; per node its frame and order
// plane; then extents, by node size: a thread per node of up to 8 leaves, a
// wave per node of up to 1,024, and above that a workgroup per 1,024 leaves
// that adds its share to every such node over them. Bound by memory latency
// at small sizes (six launches) and by the triangle reads of the mid sizes at
// large ones. The large nodes matter: with axis-aligned boxes above 512
// leaves the 1.3M-triangle walk takes twice the steps.
#include <algorithm>

#include "axsq_cull.hpp"
#include "axsq_internal.hpp"

namespace axsq {

namespace {

constexpr int kSmallNode = 8;
constexpr int kLargeNode = 1024;
constexpr int kMaxLargePath = 256;  // large nodes over one 1,024-leaf chunk
constexpr int kCullWave = 64;
constexpr int kClassSamples = 256;
// ctl: [0] unusable, [1] [2] list lengths; k_cull_class: [3] loose samples, [4 + k]
// and [8 + k] nodes of size k whose boxes are over 2 and 1.5 times as thick, [12]
// joined samples
constexpr int kCullCtl = 16;

__device__ __forceinline__ void mesh_coords(const CullSpace& cs, const double* V, float x[3]) {
  for (int d = 0; d < 3; ++d) x[d] = (float)((V[d] - cs.o[d]) * cs.scale);
}

struct Extents {
  float lo[3], hi[3];
  __device__ __forceinline__ void clear() {
    for (int d = 0; d < 3; ++d) {
      lo[d] = INFINITY;
      hi[d] = -INFINITY;
    }
  }
  __device__ __forceinline__ void add(const float t[3], float e) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      lo[d] = fminf(lo[d], t[d] - e);
      hi[d] = fmaxf(hi[d], t[d] + e);
    }
  }
  __device__ __forceinline__ void merge(const Extents& o) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      lo[d] = fminf(lo[d], o.lo[d]);
      hi[d] = fmaxf(hi[d], o.hi[d]);
    }
  }
};

// The share of a vertex at x; tau in mesh coordinates. A projection is off by
// 2^-24 |x| (x itself) and 4 2^-24 |p| (axsq_cull.hpp), t - e by 2^-24 |t| more.
__device__ __forceinline__ void add_vertex(const CullNode& n, const float x[3], float tau,
                                           Extents& out) {
  float t[3];
  cull_project(n.w, n.u, n.m, x, t);
  const float e = fmaf(fabsf(t[0]) + fabsf(t[1]) + fabsf(t[2]), 3.3e-7f, tau);
  out.add(t, fmaf(fabsf(x[0]) + fabsf(x[1]) + fabsf(x[2]), 6.6e-8f, e));
}

// Adds leaf pos's triangle records to the extents.
template <bool CELLS>
__device__ __forceinline__ void add_leaf(const CullNode& n, const CullSpace& cs,
                                         const TriRec* __restrict__ tris,
                                         const float* __restrict__ tau, int32_t pos, Extents& out) {
  const float t = tau[pos];
  const int nrec = CELLS ? tris[2 * (int64_t)pos].pad : 1;
  for (int e = 0; e < nrec; ++e) {
    const double* T = tris[CELLS ? 2 * (int64_t)pos + e : (int64_t)pos].v;
    for (int k = 0; k < 3; ++k) {
      float x[3];
      mesh_coords(cs, T + 3 * k, x);
      add_vertex(n, x, t, out);
    }
  }
}

// How far a triangle's computed closest point can lie from the triangle, for
// queries up to `reach` away; negative when no useful bound holds.
//  - Face: the weights are ratios of differences of products of dot products.
//    A dot product of an edge (at most L) with a difference to the query (at
//    most R) is off by 5 u L R, a difference of two products by 22 u (L R)^2,
//    the denominator |n|^2 by 70 u (L R)^2 (u = 2^-53), so the point is off by
//    less than 256 u L (L R)^2 / |n|^2 where that ratio is well below 1.
//  - Edge: the region tests allow 1e-12 (SignedDistance.hpp:647), so the
//    parameter can leave [0, 1] by (1e-12 + 16 u L R) / |e|^2.
// A triangle with two equal corners has |n| = 0 and never takes the face
// branch: the equal dot products send it to an edge or a vertex.
__device__ __forceinline__ float tri_tau(const double T[9], double reach) {
  double e2[3], lmax = 0.0, emin = kDblMax;
  bool same = false;
  for (int k = 0; k < 3; ++k) {
    const double* A = T + 3 * k;
    const double* B = T + 3 * ((k + 1) % 3);
    const double d0 = B[0] - A[0], d1 = B[1] - A[1], d2 = B[2] - A[2];
    e2[k] = d0 * d0 + d1 * d1 + d2 * d2;
    const bool eq = A[0] == B[0] && A[1] == B[1] && A[2] == B[2];
    same = same || eq;
    lmax = fmax(lmax, e2[k]);
    if (!eq) emin = fmin(emin, e2[k]);
  }
  if (!(lmax < 1e30)) return -1.0f;  // also NaN corners
  if (lmax == 0.0) return 0.0f;      // a point
  if (!(emin >= 4e-12)) return -1.0f;
  const double L = sqrt(lmax), LR = L * reach;
  double tau = (1.1e-12 + 1.8e-15 * LR) / sqrt(emin);
  if (!same) {
    double n[3];
    tri_normal(T, n);
    const double S = n[0] * n[0] + n[1] * n[1] + n[2] * n[2];
    const double rho = 2.9e-14 * LR * LR / S;
    if (!(rho <= 0.25)) return -1.0f;
    tau += rho * L;
  }
  return (float)(tau * 1.000001);
}

// Per leaf: tau, its triangles' NormRec (norms given), and the running sum of
// normals within its block of 256.
template <bool CELLS>
__global__ __launch_bounds__(kBlock) void k_cull_leaf(const TriRec* __restrict__ tris, int64_t n,
                                                       double reach, double tau_max, double scale,
                                                       float* __restrict__ tau,
                                                       double* __restrict__ pre,
                                                       double* __restrict__ totals,
                                                       NormRec* __restrict__ norms,
                                                       int32_t* __restrict__ ctl) {
  __shared__ double s_w[kBlock / kCullWave][3];
  const int64_t pos = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  double nr[3] = {0.0, 0.0, 0.0};
  if (pos < n) {
    float t = 0.0f;
    const int nrec = CELLS ? tris[2 * pos].pad : (tris[pos].id >= 0 ? 1 : 0);
    for (int e = 0; e < nrec; ++e) {
      double T[9], m[3];
      for (int k = 0; k < 9; ++k) T[k] = tris[CELLS ? 2 * pos + e : pos].v[k];
      const float te = tri_tau(T, reach);
      t = (te < 0.0f || t < 0.0f) ? -1.0f : fmaxf(t, te);
      tri_normal(T, m);
      for (int d = 0; d < 3; ++d) nr[d] += m[d];
      if (norms) {
        NormRec r;
        unit3(m, r.un);
        const bool flat = tri_degenerate(m);
        for (int k = 0; k < 3; ++k) r.angle[k] = flat ? -1.0 : tri_angle(T, k);
        norms[CELLS ? 2 * pos + e : pos] = r;
      }
    }
    if (!(t >= 0.0f && t <= tau_max)) {
      atomicOr(&ctl[0], 1);
      t = 0.0f;
      for (int d = 0; d < 3; ++d) nr[d] = 0.0;
    }
    tau[pos] = (float)((double)t * scale * 1.000001);
  }
  const int lane = (int)threadIdx.x % kCullWave, wv = (int)threadIdx.x / kCullWave;
  for (int o = 1; o < kCullWave; o <<= 1)
    for (int d = 0; d < 3; ++d) {
      const double v = __shfl_up(nr[d], o);
      if (lane >= o) nr[d] += v;
    }
  if (lane == kCullWave - 1)
    for (int d = 0; d < 3; ++d) s_w[wv][d] = nr[d];
  __syncthreads();
  for (int k = 0; k < wv; ++k)
    for (int d = 0; d < 3; ++d) nr[d] += s_w[k][d];
  if (pos < n)
    for (int d = 0; d < 3; ++d) pre[3 * pos + d] = nr[d];
  if (threadIdx.x == kBlock - 1)
    for (int d = 0; d < 3; ++d) totals[3 * (int64_t)blockIdx.x + d] = nr[d];
}

// Exclusive sums of the block totals, one block.
__global__ __launch_bounds__(1024) void k_cull_scan(double* __restrict__ totals, int64_t nb) {
  __shared__ double s[2][3][1024];
  double base[3] = {0.0, 0.0, 0.0};
  const int t = (int)threadIdx.x;
  for (int64_t b0 = 0; b0 < nb; b0 += 1024) {
    const int64_t b = b0 + t;
    double own[3];
    for (int d = 0; d < 3; ++d) own[d] = b < nb ? totals[3 * b + d] : 0.0;
    int cur = 0;
    for (int d = 0; d < 3; ++d) s[0][d][t] = own[d];
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
      for (int d = 0; d < 3; ++d)
        s[1 - cur][d][t] = s[cur][d][t] + (t >= o ? s[cur][d][t - o] : 0.0);
      cur = 1 - cur;
      __syncthreads();
    }
    if (b < nb)
      for (int d = 0; d < 3; ++d) totals[3 * b + d] = base[d] + s[cur][d][t] - own[d];
    for (int d = 0; d < 3; ++d) base[d] += s[cur][d][1023];
    __syncthreads();
  }
}

// The unit mean normal of a node's triangles, from the prefix sums (pre within
// blocks, base over them); x where it vanishes.
__device__ __forceinline__ void mean_normal(const Node64& nd, const double* __restrict__ pre,
                                            const double* __restrict__ base, double w[3]) {
  double len = 0.0;
  for (int d = 0; d < 3; ++d) {
    const double hi = pre[3 * (int64_t)nd.hi + d] + base[3 * (int64_t)(nd.hi / kBlock) + d];
    const double lo = nd.lo > 0 ? pre[3 * (int64_t)(nd.lo - 1) + d] +
                                      base[3 * (int64_t)((nd.lo - 1) / kBlock) + d]
                                : 0.0;
    w[d] = hi - lo;
    len += w[d] * w[d];
  }
  const double il = len > 0.0 ? 1.0 / sqrt(len) : 0.0;
  if (il > 0.0 && il < 1e300) {
    for (int d = 0; d < 3; ++d) w[d] *= il;
  } else {
    w[0] = 1.0;
    w[1] = w[2] = 0.0;
  }
}

// What oriented boxes gain on this mesh, from the nodes over kClassSamples leaves
// spread over the tree: four waves each descend to the node of at most 32,768,
// 4,096, 512 and 64 leaves over such a leaf and compare the extent of the
// axis-aligned box along the mean normal with that of what the node holds,
// tolerances included (of larger nodes 1,024 leaves are looked at). A sample is
// loose where most leaves' tolerances are more than a quarter of their triangles'
// height, joined where most of its 64 triangles share a corner with another one.
// Bound by latency: a descent of up to 16 dependent loads, 16 leaf loads a lane.
template <bool CELLS>
__global__ __launch_bounds__(4 * kCullWave) void k_cull_class(CullSpace cs,
                                                               const Node64* __restrict__ nodes,
                                                               int32_t ninner,
                                                               const TriRec* __restrict__ tris,
                                                               const float* __restrict__ tau,
                                                               const double* __restrict__ pre,
                                                               const double* __restrict__ base,
                                                               int32_t* __restrict__ ctl) {
  const int lane = (int)threadIdx.x % kCullWave, k = (int)threadIdx.x / kCullWave;
  const int32_t p = (int32_t)((2 * (int64_t)blockIdx.x + 1) * (ninner + 1) / (2 * kClassSamples));
  const int32_t cap = 32768 >> (3 * k);
  Node64 nd = nodes[0];
  while (nd.hi - nd.lo + 1 > cap) {  // a child holds fewer leaves
    const int32_t next = p <= nd.mid ? nd.lc : nd.rc;
    if (next < 0 || next >= ninner) break;
    nd = nodes[next];
  }
  double w[3];
  mean_normal(nd, pre, base, w);
  const int32_t size = nd.hi - nd.lo + 1, step = (size + 1023) / 1024;
  double lo = INFINITY, hi = -INFINITY;
  int32_t loose = 0, seen = 0;
#pragma unroll 4
  for (int32_t q = nd.lo + lane * step; q <= nd.hi; q += kCullWave * step) {
    const double e = tau[q];
    const int nrec = CELLS ? tris[2 * (int64_t)q].pad : 1;
    for (int r = 0; r < nrec; ++r) {
      const double* T = tris[CELLS ? 2 * (int64_t)q + r : (int64_t)q].v;
      double l2 = 0.0;
      for (int c = 0; c < 3; ++c) {
        double t = 0.0, d2 = 0.0;
        for (int d = 0; d < 3; ++d) {
          t += (T[3 * c + d] - cs.o[d]) * cs.scale * w[d];
          const double g = T[(3 * c + 3 + d) % 9] - T[3 * c + d];
          d2 += g * g;
        }
        lo = fmin(lo, t - e);
        hi = fmax(hi, t + e);
        l2 = fmax(l2, d2);
      }
      double m[3];
      tri_normal(T, m);
      const double h = sqrt((m[0] * m[0] + m[1] * m[1] + m[2] * m[2]) / l2) * cs.scale;
      ++seen;
      loose += e > 0.25 * h;
    }
  }
  for (int o = kCullWave / 2; o > 0; o >>= 1) {
    lo = fmin(lo, __shfl_xor(lo, o));
    hi = fmax(hi, __shfl_xor(hi, o));
    loose += __shfl_xor(loose, o);
    seen += __shfl_xor(seen, o);
  }
  double box = 0.0;
  for (int d = 0; d < 3; ++d) {
    const double l0 = (nd.flags & 1) ? nd.l[d] : nd.r[d], l1 = (nd.flags & 1) ? nd.l[3 + d] : nd.r[3 + d];
    const double r0 = (nd.flags & 2) ? nd.r[d] : l0, r1 = (nd.flags & 2) ? nd.r[3 + d] : l1;
    box += fabs(w[d]) * (fmax(l1, r1) - fmin(l0, r0)) * cs.scale;
  }
  // the walk's slack on both sides: ties, and projections at a unit's distance
  const double own = hi - lo + 2e-6 * (cs.scale + 1.0);
  if (lane == 0 && box > 2.0 * own) atomicAdd(&ctl[4 + k], 1);
  if (lane == 0 && box > 1.5 * own) atomicAdd(&ctl[8 + k], 1);
  if (k < 3) return;
  // at most 64 leaves, one a lane
  const bool has = lane < size;
  const int32_t q = nd.lo + (has ? lane : 0);
  const double* T = tris[CELLS ? 2 * (int64_t)q : (int64_t)q].v;
  double v[9];
  for (int c = 0; c < 9; ++c) v[c] = T[c];
  bool meets = false;
  const int32_t held = min(size, kCullWave);
  for (int o = 0; o < held; ++o)
    for (int c = 0; c < 9; c += 3) {
      const double x = __shfl(v[c], o), y = __shfl(v[c + 1], o), z = __shfl(v[c + 2], o);
      const bool eq = (x == v[0] && y == v[1] && z == v[2]) ||
                      (x == v[3] && y == v[4] && z == v[5]) ||
                      (x == v[6] && y == v[7] && z == v[8]);
      meets = meets || (o != lane && eq);
    }
  const int32_t shared = __popcll(__ballot(has && meets));
  if (lane == 0 && 2 * loose > seen) atomicAdd(&ctl[3], 1);
  if (lane == 0 && 2 * shared > held) atomicAdd(&ctl[12], 1);
}

__device__ __forceinline__ uint32_t ordered(float f) {
  const uint32_t b = __float_as_uint(f);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float unordered(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

__device__ __forceinline__ void store_extents(CullNode* __restrict__ n, const Extents& l,
                                              const Extents& r, int32_t flags) {
  constexpr uint32_t kNone = 0xfc007c00u;  // an invalid child: from +inf to -inf
  for (int d = 0; d < 3; ++d) {
    n->l[d] = (flags & 1) ? half_range(l.lo[d], l.hi[d]) : kNone;
    n->r[d] = (flags & 2) ? half_range(r.lo[d], r.hi[d]) : kNone;
  }
}

// Per node: frame, order plane and links; extents of nodes of at most 8
// leaves; the others are listed by size. ctl[1], ctl[2]: list lengths. A large
// node's place in its list is kept in l[0] until k_cull_large_end.
template <bool CELLS>
__global__ __launch_bounds__(kBlock) void k_cull_nodes(CullSpace cs,
                                                        const Node64* __restrict__ nodes,
                                                        int32_t ninner,
                                                        const TriRec* __restrict__ tris,
                                                        const float* __restrict__ tau,
                                                        const double* __restrict__ pre,
                                                        const double* __restrict__ base,
                                                        CullNode* __restrict__ out,
                                                        int32_t* __restrict__ mid_list,
                                                        int32_t* __restrict__ large_list,
                                                        uint32_t* __restrict__ acc,
                                                        int32_t* __restrict__ ctl) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  bool mid = false, large = false;
  if (i < ninner) {
    const Node64 nd = nodes[i];
    CullNode n;
    n.lc = nd.lc;
    n.rc = nd.rc;
    double w[3];
    mean_normal(nd, pre, base, w);
    double cl[3], cr[3], D[3], dl = 0.0, tw = 0.0;
    for (int d = 0; d < 3; ++d) {  // centroids as in BoxTests::right_first
      cl[d] = 0.5 * (nd.l[d] + nd.l[3 + d]);
      cr[d] = 0.5 * (nd.r[d] + nd.r[3 + d]);
      D[d] = cr[d] - cl[d];
      dl += D[d] * D[d];
      tw += D[d] * w[d];
    }
    // second axis: the split direction in the tangent plane
    double u[3], ul = 0.0;
    for (int d = 0; d < 3; ++d) {
      u[d] = D[d] - tw * w[d];
      ul += u[d] * u[d];
    }
    const bool split = ul > 1e-12 * dl && ul > 0.0 && ul < 1e300;
    if (split) {
      const double iu = 1.0 / sqrt(ul);
      for (int d = 0; d < 3; ++d) u[d] *= iu;
    } else {  // any tangent: the axis least along w, made orthogonal; no order
              // plane, D has a third component in this frame
      const int k = fabs(w[0]) <= fabs(w[1]) ? (fabs(w[0]) <= fabs(w[2]) ? 0 : 2)
                                             : (fabs(w[1]) <= fabs(w[2]) ? 1 : 2);
      const double wk = k == 0 ? w[0] : k == 1 ? w[1] : w[2];
      double m = 0.0;
      for (int d = 0; d < 3; ++d) {
        u[d] = (d == k ? 1.0 : 0.0) - wk * w[d];
        m += u[d] * u[d];
      }
      const double iu = 1.0 / sqrt(m);
      for (int d = 0; d < 3; ++d) u[d] *= iu;
    }
    const double dlen = sqrt(dl), idl = dl > 0.0 ? 1.0 / dlen : 0.0;
    const bool plane = split && idl > 0.0 && idl < 1e30;
    double a = 0.0, bb = 0.0;
    for (int d = 0; d < 3; ++d) {
      n.w[d] = (float)w[d];
      n.u[d] = (float)u[d];
      n.m[d] = (float)((0.5 * (cl[d] + cr[d]) - cs.o[d]) * cs.scale);
      a += D[d] * idl * w[d];
      bb += D[d] * idl * u[d];
    }
    n.a = plane ? (float)a : 0.0f;
    n.b = plane ? (float)bb : 0.0f;
    n.inv_d = plane ? (float)(idl / cs.scale * 1.000001) : INFINITY;
    Extents xl, xr;
    xl.clear();
    xr.clear();
    const int32_t size = nd.hi - nd.lo + 1;
    large = size > kLargeNode;
    mid = !large && size > kSmallNode;
    if (!large && !mid) {
      for (int32_t p = nd.lo; p <= nd.hi; ++p)
        add_leaf<CELLS>(n, cs, tris, tau, p, p <= nd.mid ? xl : xr);
    }
    store_extents(&n, xl, xr, nd.flags);
    out[i] = n;
  }
  // list entries, one atomic per wave and list
  const int lane = (int)threadIdx.x % kCullWave;
  const uint64_t below = lane == 0 ? 0ull : (~0ull >> (kCullWave - lane));
  for (int k = 0; k < 2; ++k) {
    const uint64_t m = __ballot(k == 0 ? mid : large);
    int32_t at = 0;
    if (lane == 0 && m) at = atomicAdd(&ctl[1 + k], __popcll(m));
    at = __shfl(at, 0);
    at += __popcll(m & below);
    if (k == 0 && mid) mid_list[at] = (int32_t)i;
    if (k == 1 && large) {
      large_list[at] = (int32_t)i;
      out[i].l[0] = (uint32_t)at;
      for (int d = 0; d < 12; ++d) acc[12 * (int64_t)at + d] = (d % 6) < 3 ? 0xffffffffu : 0u;
    }
  }
}

__device__ __forceinline__ void wave_reduce(Extents& x) {
  for (int o = kCullWave / 2; o > 0; o >>= 1)
    for (int d = 0; d < 3; ++d) {
      x.lo[d] = fminf(x.lo[d], __shfl_xor(x.lo[d], o));
      x.hi[d] = fmaxf(x.hi[d], __shfl_xor(x.hi[d], o));
    }
}

// One wave per node of 9 to 1,024 leaves; the list's length is on the device,
// so a fixed grid strides over it.
template <bool CELLS>
__global__ __launch_bounds__(kBlock) void k_cull_mid(CullSpace cs,
                                                      const Node64* __restrict__ nodes,
                                                      const TriRec* __restrict__ tris,
                                                      const float* __restrict__ tau,
                                                      const int32_t* __restrict__ list,
                                                      const int32_t* __restrict__ ctl,
                                                      CullNode* __restrict__ out) {
  const int lane = (int)threadIdx.x % kCullWave;
  const int32_t waves = (int32_t)(gridDim.x * (kBlock / kCullWave));
  const int32_t count = ctl[1];
  for (int32_t j = (int32_t)(blockIdx.x * (kBlock / kCullWave) + threadIdx.x / kCullWave);
       j < count; j += waves) {
    const int32_t i = list[j];
    const int32_t lo = nodes[i].lo, hi = nodes[i].hi, split = nodes[i].mid;
    const CullNode n = out[i];
    Extents xl, xr;
    xl.clear();
    xr.clear();
    for (int32_t p = lo + lane; p <= hi; p += kCullWave) {
      Extents x;
      x.clear();
      add_leaf<CELLS>(n, cs, tris, tau, p, x);
      if (p <= split)
        xl.merge(x);
      else
        xr.merge(x);
    }
    wave_reduce(xl);
    wave_reduce(xr);
    if (lane == 0) store_extents(out + i, xl, xr, nodes[i].flags);
  }
}

// One workgroup per 1,024 leaves: its share of every larger node over them,
// from vertices held in registers (a node costs no triangle reads: for 2.1M
// triangles the kernel took 1.14 ms reading them per node). A node's share on
// one side of its split only, the common case, reduces that side alone.
template <bool CELLS>
__global__ __launch_bounds__(kBlock) void k_cull_large(CullSpace cs,
                                                        const Node64* __restrict__ nodes,
                                                        int32_t ninner,
                                                        const TriRec* __restrict__ tris,
                                                        const float* __restrict__ tau,
                                                        const CullNode* __restrict__ out,
                                                        uint32_t* __restrict__ acc,
                                                        int32_t* __restrict__ ctl) {
  constexpr int kPer = kLargeNode / kBlock;  // leaves per thread
  constexpr int kVerts = CELLS ? 6 : 3;
  __shared__ int32_t s_list[kMaxLargePath];
  __shared__ int32_t s_n;
  const int32_t a = (int32_t)blockIdx.x * kLargeNode;
  const int32_t b = min(a + kLargeNode - 1, ninner);
  if (threadIdx.x == 0) {  // from the root down: list doubles as the stack's record
    int32_t n = 0, done = 0;
    bool full = false;
    if (ninner + 1 > kLargeNode) s_list[n++] = 0;
    while (done < n) {
      const Node64& nd = nodes[s_list[done++]];
      const int32_t c[2] = {nd.lc, nd.rc};
      const int32_t lo[2] = {nd.lo, nd.mid + 1}, hi[2] = {nd.mid, nd.hi};
      for (int k = 0; k < 2; ++k) {
        if (c[k] < 0 || c[k] >= ninner || hi[k] < a || lo[k] > b) continue;
        if (hi[k] - lo[k] + 1 <= kLargeNode) continue;
        if (n < kMaxLargePath)
          s_list[n++] = c[k];
        else
          full = true;
      }
    }
    if (full) atomicOr(&ctl[0], 1);
    s_n = n;
  }
  float x[kPer][kVerts][3], t[kPer];
  int nv[kPer];
  for (int j = 0; j < kPer; ++j) {
    const int32_t p = a + j * kBlock + (int32_t)threadIdx.x;
    nv[j] = 0;
    t[j] = 0.0f;
    for (int k = 0; k < kVerts; ++k)
      for (int d = 0; d < 3; ++d) x[j][k][d] = 0.0f;
    if (p <= b) {
      t[j] = tau[p];
      nv[j] = CELLS ? 3 * tris[2 * (int64_t)p].pad : 3;
      for (int k = 0; k < kVerts; ++k)
        if (k < nv[j]) {
          const int64_t rec = CELLS ? 2 * (int64_t)p + k / 3 : (int64_t)p;
          mesh_coords(cs, tris[rec].v + 3 * (k % 3), x[j][k]);
        }
    }
  }
  __syncthreads();
  const int lane = (int)threadIdx.x % kCullWave;
  for (int32_t i = 0; i < s_n; ++i) {
    const CullNode n = out[s_list[i]];
    const int32_t lo = nodes[s_list[i]].lo, hi = nodes[s_list[i]].hi, split = nodes[s_list[i]].mid;
    uint32_t* to = acc + 12 * (int64_t)n.l[0];
    for (int side = 0; side < 2; ++side) {
      const int32_t from = side == 0 ? max(lo, a) : max(split + 1, a);
      const int32_t last = side == 0 ? min(split, b) : min(hi, b);
      if (from > last) continue;  // uniform
      Extents e;
      e.clear();
      for (int j = 0; j < kPer; ++j) {
        const int32_t p = a + j * kBlock + (int32_t)threadIdx.x;
        if (p < from || p > last) continue;
        for (int k = 0; k < kVerts; ++k)
          if (k < nv[j]) add_vertex(n, x[j][k], t[j], e);
      }
      wave_reduce(e);
      if (lane == 0) {
        for (int d = 0; d < 3; ++d) {
          if (e.lo[d] <= e.hi[d]) {
            atomicMin(to + 6 * side + d, ordered(e.lo[d]));
            atomicMax(to + 6 * side + 3 + d, ordered(e.hi[d]));
          }
        }
      }
    }
  }
}

__global__ __launch_bounds__(kBlock) void k_cull_large_end(const Node64* __restrict__ nodes,
                                                            const int32_t* __restrict__ list,
                                                            const int32_t* __restrict__ ctl,
                                                            const uint32_t* __restrict__ acc,
                                                            CullNode* __restrict__ out) {
  const int32_t count = ctl[2];
  for (int32_t j = (int32_t)(blockIdx.x * blockDim.x + threadIdx.x); j < count;
       j += (int32_t)(gridDim.x * blockDim.x)) {
    Extents x[2];
    for (int side = 0; side < 2; ++side)
      for (int d = 0; d < 3; ++d) {
        x[side].lo[d] = unordered(acc[12 * (int64_t)j + 6 * side + d]);
        x[side].hi[d] = unordered(acc[12 * (int64_t)j + 6 * side + 3 + d]);
      }
    store_extents(out + list[j], x[0], x[1], nodes[list[j]].flags);
  }
}

template <bool CELLS>
int build(const axsq_bvh* b, const TriRec* tris, const CullSpace& cs, double diag, int parts,
          CullNode* out, NormRec* norms, CullResult* res, Workspace& ws, hipStream_t s) {
  const int64_t n = b->n;
  const int32_t ninner = (int32_t)(n - 1);
  const int64_t nb = grid_for(n);
  AXSQ_TRY(ws.k0.ensure(sizeof(float) * (size_t)n));
  AXSQ_TRY(ws.k1.ensure(sizeof(int32_t) * (size_t)ninner));
  AXSQ_TRY(ws.v0.ensure(sizeof(double) * 3 * (size_t)n));
  AXSQ_TRY(ws.v1.ensure(sizeof(double) * 3 * (size_t)nb));
  AXSQ_TRY(ws.cnt.ensure(sizeof(int32_t) * kCullCtl));
  float* tau = ws.k0.as<float>();
  double* pre = ws.v0.as<double>();
  double* totals = ws.v1.as<double>();
  int32_t* ctl = ws.cnt.as<int32_t>();
  if (parts & kCullLeaves) {
    AXSQ_TRY(fill_i32(ctl, 0, kCullCtl, s));
    k_cull_leaf<CELLS><<<(unsigned)nb, kBlock, 0, s>>>(tris, n, kCullReach * diag,
                                                       diag * (1.0 / 1024.0), cs.scale, tau, pre,
                                                       totals, norms, ctl);
    AXSQ_CHECK_HIP(hipGetLastError());
    k_cull_scan<<<1, 1024, 0, s>>>(totals, nb);
    AXSQ_CHECK_HIP(hipGetLastError());
  }
  if (parts & kCullClass) {
    k_cull_class<CELLS><<<kClassSamples, 4 * kCullWave, 0, s>>>(cs, b->nodes, ninner, tris, tau, pre,
                                                            totals, ctl);
    AXSQ_CHECK_HIP(hipGetLastError());
  }
  if (parts & kCullBoxes) {
    int32_t* mid_list = ws.k1.as<int32_t>();
    // nodes over 1,024 leaves: few in a balanced tree, up to ninner - 1,023 in a
    // chain, each with 12 running extents
    const size_t nlarge = (size_t)std::max<int64_t>((int64_t)ninner - kLargeNode + 1, 1);
    AXSQ_TRY(ws.redo.ensure(sizeof(int32_t) * nlarge));
    AXSQ_TRY(ws.misc.ensure(sizeof(uint32_t) * 12 * nlarge));
    int32_t* large_list = ws.redo.as<int32_t>();
    uint32_t* acc = ws.misc.as<uint32_t>();
    k_cull_nodes<CELLS><<<grid_for(ninner), kBlock, 0, s>>>(cs, b->nodes, ninner, tris, tau, pre,
                                                            totals, out, mid_list, large_list,
                                                            acc, ctl);
    AXSQ_CHECK_HIP(hipGetLastError());
    if (n > kSmallNode) {
      const unsigned g = (unsigned)std::min<int64_t>((n / 6 + 3) / 4 + 1, 8192);
      k_cull_mid<CELLS><<<g, kBlock, 0, s>>>(cs, b->nodes, tris, tau, mid_list, ctl, out);
      AXSQ_CHECK_HIP(hipGetLastError());
    }
    if (n > kLargeNode) {
      k_cull_large<CELLS><<<(unsigned)((n + kLargeNode - 1) / kLargeNode), kBlock, 0, s>>>(
          cs, b->nodes, ninner, tris, tau, out, acc, ctl);
      AXSQ_CHECK_HIP(hipGetLastError());
      k_cull_large_end<<<(unsigned)std::min<int64_t>(n / kLargeNode / kBlock + 1, 256), kBlock, 0,
                         s>>>(b->nodes, large_list, ctl, acc, out);
      AXSQ_CHECK_HIP(hipGetLastError());
    }
  }
  int32_t h[kCullCtl];
  AXSQ_CHECK_HIP(hipMemcpyAsync(h, ctl, sizeof(h), hipMemcpyDeviceToHost, s));
  AXSQ_CHECK_HIP(hipStreamSynchronize(s));
  res->bad = h[0] != 0;
  // Of a curved, tilted or gently uneven surface nearly every node of some size is
  // less than half as thick as its box. Of a flat one along the axes, or of a
  // rough one whose parts are as thick as their boxes at any size, none is. In
  // between lie strong noise on a curved ground, whose larger nodes are thinner by
  // half, and large flat facets along the axes, where only those over an edge are;
  // the small nodes tell these apart. Nodes over 2x at 64, 512, 4,096 leaves / over
  // 1.5x at 4,096, 32,768 / over 1.5x at 64, per cent:
  //   spheres, tori, hills, tilted planes   100 90-100 57-100
  //   noise of 1/20 on a sphere              4  0 44 /  88 100 / 30
  //   noise of 12 cells on hills             0  0  0 /  26  82 / 26
  //   height fields with noise               0  0  0 /   0 0-6 / 11-20
  //   cubes, 196,608 and 786,432             0  0  4 / 46-63 100 / 7-12
  //   flat along the axes                    0  0  0 /   0   0 / 0
  // Triangles at random (0 0 0 / 0 0 / 16) are another matter: they fill space, and
  // most queries are near one.
  const int third = kClassSamples / 3;
  const bool thin = std::max({h[5], h[6], h[7]}) > third;
  const bool uneven = std::max(h[8], h[9]) > third && 5 * h[11] > kClassSamples;
  const bool joined = 2 * h[12] > kClassSamples;
  res->plain = joined && !thin && !uneven;
  res->flat = res->plain && 50 * h[11] < kClassSamples;
  res->crowd = !joined && !thin;
  res->loose = 2 * h[3] > kClassSamples && h[7] <= third;
  return AXSQ_OK;
}

}  // namespace

int cull_build(const axsq_bvh* b, const TriRec* tris, bool cells, const CullSpace& cs, double diag,
               int parts, CullNode* out, NormRec* norms, CullResult* res, hipStream_t s) {
  Workspace& ws = workspace();
  return cells ? build<true>(b, tris, cs, diag, parts, out, norms, res, ws, s)
               : build<false>(b, tris, cs, diag, parts, out, norms, res, ws, s);
}

}  // namespace axsq
