// axsq_mesh.hip -- triangle-triangle intersection and the BVH mesh
// self-intersection test (quest::findTriMeshIntersectionsBVH) for gfx950.
//
// The reference (quest/detail/MeshTester_detail.hpp:159-341) builds corner
// boxes and degenerate flags, a BVH over the boxes, runs findBoundingBoxes
// for every box (count, scan, fill of all candidates), keeps the pairs i < j
// and tests them. Here the triangle test is the traversal's leaf action
// (the custom leaf action of quest/examples/quest_bvh_two_pass.cpp:144-232): a wave
// walks for the triangles at neighbouring leaves, meets each pair once, from its
// lower leaf, and tests it on the spot, keeping kPairSlots hits of the smaller
// index. A scan of the hit counts places every triangle's pairs; triangles with
// more hits walk again to write them all. The candidate lists are never stored
// (the walk's own list, of leaves and triangles, is in LDS). The output
// order is the sequential path's: pairs grouped by the first triangle, the
// second in the first's BVH traversal order; degenerate indices ascending.
#include <hip/hip_runtime.h>

#include "axsq_internal.hpp"
#include "axsq_traverse.hpp"
#include "axsq_tritri.hpp"

namespace axsq {
namespace {

__device__ __forceinline__ V3 load_v3(const double* p) { return {p[0], p[1], p[2]}; }

// The vertices as 32-byte records, for k_tri_setup's gathers: three arrays of
// coordinates cost a line each.
__global__ __launch_bounds__(kBlock) void k_pack_verts(const double* __restrict__ x,
                                                       const double* __restrict__ y,
                                                       const double* __restrict__ z, int64_t n,
                                                       double2* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  out[2 * i] = make_double2(x[i], y[i]);
  out[2 * i + 1] = make_double2(z[i], 0.0);
}

// Triangle corners (A B C, TriRec), the corner box (BoundingBox{A, B, C},
// compute_bounding_box.hpp:110-114, BoundingBox.hpp:405-422,464-482) and the
// degenerate flag (Triangle::degenerate, Triangle.hpp:104-109,327-330). verts:
// k_pack_verts' records, or NULL. A triangle that refers to a vertex outside
// [0, nverts) sets bit 1 of *status and gets an invalid box: taken at vertex 0,
// a connectivity of such triangles would be as many boxes on one point, and the
// walk test all their pairs before the call ends with the error.
// 2.6M triangles of 1.3M vertices: 247 us from the three arrays, 186 with the
// records (15 of it making them).
__global__ __launch_bounds__(kBlock) void k_tri_setup(const double* __restrict__ x,
                                                      const double* __restrict__ y,
                                                      const double* __restrict__ z,
                                                      const double2* __restrict__ verts,
                                                      const int32_t* __restrict__ conn,
                                                      int64_t n, int64_t nverts,
                                                      TriRec* __restrict__ tri,
                                                      double* __restrict__ boxes,
                                                      int32_t* __restrict__ degen,
                                                      int32_t* __restrict__ npair,
                                                      int32_t* __restrict__ status) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  TriRec r;
  double* t = r.v;
  bool bad = false;
  for (int k = 0; k < 3; ++k) {
    int32_t v = conn[3 * c + k];
    if (v < 0 || v >= nverts) {
      bad = true;
      v = 0;
    }
    if (verts) {
      const double2 a = verts[2 * (int64_t)v], b = verts[2 * (int64_t)v + 1];
      t[3 * k] = a.x;
      t[3 * k + 1] = a.y;
      t[3 * k + 2] = b.x;
    } else {
      t[3 * k] = x[v];
      t[3 * k + 1] = y[v];
      t[3 * k + 2] = z[v];
    }
  }
  double b[6] = {t[0], t[1], t[2], t[0], t[1], t[2]};
  for (int corner = 1; corner < 3; ++corner)
    for (int d = 0; d < 3; ++d) {
      const double p = t[3 * corner + d];
      if (p < b[d]) b[d] = p;
      if (p > b[3 + d]) b[3 + d] = p;
    }
  if (bad) {
    atomicOr(status, 2);
    for (int d = 0; d < 3; ++d) {
      b[d] = kDblMax;
      b[3 + d] = -kDblMax;
    }
  }
  double nrm[3];
  tri_normal(t, nrm);
  degen[c] = tri_degenerate(nrm) ? 1 : 0;
  npair[c] = 0;
  r.id = (int32_t)c;
  r.pad = 0;
  tri[c] = r;
  double2* o = reinterpret_cast<double2*>(boxes + 6 * c);
  for (int k = 0; k < 3; ++k) o[k] = make_double2(b[2 * k], b[2 * k + 1]);
}

constexpr int kPairSlots = 4;  // hits kept per triangle by the first walk

struct IsectArgs {
  const Node64* nodes;
  const FindNode* fnodes;  // compact nodes (axsq_find.hpp) and their coordinates
  FindSpace space;
  int32_t ninner;
  const int32_t* leaf_ids;
  const double* leaf_boxes;
  const TriRec* tri;    // per triangle
  const double* boxes;  // 6 doubles per triangle (the unscaled corner box)
  int64_t n;
  double eps;
  int32_t* npair;  // hits per triangle
  int32_t* slots;  // kPairSlots per triangle: the hits' leaf positions
  const int32_t* poff;
  int32_t* first;  // entry k of a pair's member at `step` * k
  int32_t* second;
  int step;
  int32_t* more;    // triangles with more hits than slots, and their number
  uint32_t* nmore;
  int32_t* status;
};

// One walk of triangle i's box through the tree (BoundingBox::intersectsWith,
// BVH.hpp:558-560, as findBoundingBoxes tests it) that calls hit(j, j's leaf
// position) for each reached triangle j > i that intersects triangle i (boundary
// excluded).
template <class Hit>
__device__ __forceinline__ void isect_walk(const IsectArgs& a, int64_t i, lds_i32* stk, Hit&& hit) {
  double prim[6];
  for (int k = 0; k < 6; ++k) prim[k] = a.boxes[6 * i + k];
  const double* ti = a.tri[i].v;
  const V3 a0 = load_v3(ti), a1 = load_v3(ti + 3), a2 = load_v3(ti + 6);
  auto no_pref = [](const auto*, const auto*) { return false; };
  const int32_t v = traverse_voted<Node64, double>(
      a.nodes, a.ninner, stk,
      [&](const double* b) {
        return (prim[3] >= b[0] && prim[0] <= b[3]) && (prim[4] >= b[1] && prim[1] <= b[4]) &&
               (prim[5] >= b[2] && prim[2] <= b[5]);
      },
      no_pref,
      [&](int32_t pos) {
        const int32_t j = a.leaf_ids[pos];
        if ((int64_t)j <= i || (int64_t)j >= a.n) return;
        const double* tj = a.tri[j].v;
        if (tri_tri_intersect(a0, a1, a2, load_v3(tj), load_v3(tj + 3), load_v3(tj + 6), false,
                              a.eps))
          hit(j, pos);
      });
  if (v < 0) atomicOr(a.status, 1);
}

// Whether triangle f's corner box meets the scaled box of triangle s, at leaf
// position sp, and the triangles intersect.
__device__ __forceinline__ bool isect_test(const IsectArgs& a, int32_t f, int32_t s, int32_t sp) {
  // 16-byte loads: the vector L1 returns one lane's a cycle, whatever they hold
  const double2* u = reinterpret_cast<const double2*>(a.boxes + 6 * (int64_t)f);
  const double2* b = reinterpret_cast<const double2*>(a.leaf_boxes + 6 * (int64_t)sp);
  const double2 u0 = u[0], u1 = u[1], u2 = u[2], b0 = b[0], b1 = b[1], b2 = b[2];
  if (!((u1.y >= b0.x && u0.x <= b1.y) && (u2.x >= b0.y && u0.y <= b2.x) &&
        (u2.y >= b1.x && u1.x <= b2.y)))
    return false;
  V3 p[2][3];
  for (int k = 0; k < 2; ++k) {
    const double2* t = reinterpret_cast<const double2*>(a.tri + (k ? s : f));
    const double2 t0 = t[0], t1 = t[1], t2 = t[2], t3 = t[3];
    p[k][0] = {t0.x, t0.y, t1.x};
    p[k][1] = {t1.y, t2.x, t2.y};
    p[k][2] = {t3.x, t3.y, reinterpret_cast<const double*>(t)[8]};
  }
  return tri_tri_intersect(p[0][0], p[0][1], p[0][2], p[1][0], p[1][1], p[1][2], false, a.eps);
}

// Walk 1 where the compact nodes cannot serve: a lane per triangle.
__global__ __launch_bounds__(kBlock) void k_isect_count(IsectArgs a) {
  __shared__ int32_t s_stack[stack_lds_words(kBlock)];
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= a.n) return;
  const int64_t i = a.n > 1 ? (int64_t)a.leaf_ids[p] : 0;
  int32_t c = 0;
  isect_walk(a, i, lane_stack_base(s_stack), [&](int32_t, int32_t pos) {
    if (c < kPairSlots) a.slots[kPairSlots * i + c] = pos;
    ++c;
  });
  a.npair[i] = c;
}

// Walk 1: count every triangle's hits, keep kPairSlots of them in any order.
// A wave takes the triangles at `tris` neighbouring leaf positions and works
// on (triangle, node) entries as k_ray_count does on rays: 64 visits a step,
// then 64 triangle tests a step, where a lane per triangle left lanes idle in
// both (a test is some hundred FP64 instructions, and a wave at a time had few).
// Each pair is met once, from its lower leaf position p: a left child whose
// positions end at or before p is skipped (the link of a left child is the last
// position of its range). Its smaller triangle index is then the first of the
// pair, the other the second, and the reference's box test, the first's corner
// box against the second's scaled one, is done as it is; the walk's query box
// contains both boxes of p, widened by 4 units in the last place of its largest
// coordinate, which covers a scaled box that rounding left inside its corner box.
// 2.6M triangles, two crossing noisy spheres: 4.1 ms with a lane per triangle
// in mesh order on the FP64 nodes, 3.4 in leaf order on the compact ones, 0.90
// here (1.04 with the tests' loads 8 bytes wide).
constexpr int kPoolTris = 64;
__global__ __launch_bounds__(kWaveLanes) void k_isect_pool(IsectArgs a, int tris) {
  __shared__ FindPool s_pool;
  __shared__ float s_q[12][kPoolTris];
  __shared__ int32_t s_id[kPoolTris];
  const int lane = (int)threadIdx.x;
  const int64_t p0 = (int64_t)blockIdx.x * tris;
  int32_t id = -1;
  if (lane < tris && p0 + lane < a.n) {
    id = a.leaf_ids[p0 + lane];
    if ((int64_t)id >= a.n) id = -1;  // the padding of a single triangle's tree
  }
  if (id >= 0) {
    const double* sb = a.leaf_boxes + 6 * (p0 + lane);
    const double* b = a.boxes + 6 * (int64_t)id;
    double prim[6];
    for (int d = 0; d < 3; ++d) {
      const double lo = b[d] < sb[d] ? b[d] : sb[d], hi = b[3 + d] > sb[3 + d] ? b[3 + d] : sb[3 + d];
      const double w = 1e-15 * fmax(fabs(lo), fabs(hi));
      prim[d] = lo - w;
      prim[3 + d] = hi + w;
    }
    FindQuery<true> q;
    q.init(a.space, prim);
    for (int d = 0; d < 3; ++d) {
      s_q[4 * d][lane] = q.lh[d];
      s_q[4 * d + 1][lane] = q.ll[d];
      s_q[4 * d + 2][lane] = q.hh[d];
      s_q[4 * d + 3][lane] = q.hl[d];
    }
    s_id[lane] = id;
  }
  const bool done = find_pooled(
      s_pool, id >= 0, a.ninner,
      [&](uint32_t node, int who, bool& in_l, bool& in_r, uint32_t& lc, uint32_t& rc) {
        FindQuery<true> q;
        for (int d = 0; d < 3; ++d) {
          q.lh[d] = s_q[4 * d][who];
          q.ll[d] = s_q[4 * d + 1][who];
          q.hh[d] = s_q[4 * d + 2][who];
          q.hl[d] = s_q[4 * d + 3][who];
        }
        float gl, gr;
        find_visit<true, 3>(a.fnodes, node, q, gl, gr, lc, rc);
        const int32_t p = (int32_t)p0 + who;
        in_l = !(gl > 0.0f) && (int32_t)(lc & kFindPos) > p;
        in_r = !(gr > 0.0f) && !((rc & kFindLeaf) && (int32_t)(rc & kFindPos) <= p);
      },
      [&](int32_t q, int who) {
        const int32_t p = (int32_t)p0 + who, ip = s_id[who], iq = a.leaf_ids[q];
        const int32_t f = ip < iq ? ip : iq, s = ip < iq ? iq : ip, sp = ip < iq ? q : p;
        if ((int64_t)s < a.n && isect_test(a, f, s, sp)) {
          const int32_t c = atomicAdd(a.npair + f, 1);
          if (c < kPairSlots) a.slots[kPairSlots * (int64_t)f + c] = sp;
        }
      });
  if (!done && lane == 0) atomicOr(a.status, 1);
}

// Write the pairs at the scanned offsets, the kept hits in leaf order, the
// walk's; triangles with more hits than slots are listed.
__global__ __launch_bounds__(kBlock) void k_isect_emit(IsectArgs a) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int32_t c = (i < a.n) ? a.npair[i] : 0;
  if (c == 0) return;
  if (c > kPairSlots) {
    a.more[atomicAdd(a.nmore, 1u)] = (int32_t)i;
    return;
  }
  const int32_t o = a.poff[i];
  const int32_t* slot = a.slots + kPairSlots * i;
  for (int32_t k = 0; k < c; ++k) {
    const int32_t pos = slot[k];
    int32_t at = o;
    for (int32_t t = 0; t < c; ++t) at += slot[t] < pos;
    a.first[(int64_t)a.step * at] = (int32_t)i;
    a.second[(int64_t)a.step * at] = a.leaf_ids[pos];
  }
}

// The listed triangles walk again and write every hit in the walk's order: a
// wave per triangle (find_ordered), since a few have very many (a lane each on
// the FP64 nodes took 277 us at the size above, a wave each 36).
__global__ __launch_bounds__(kWaveLanes) void k_isect_more(IsectArgs a) {
  __shared__ uint32_t s_item[kOrderedItems];
  const uint32_t n = *a.nmore;
  for (uint32_t e = blockIdx.x; e < n; e += gridDim.x) {
    const int32_t i = a.more[e], o = a.poff[i], c = a.npair[i];
    FindQuery<true> q;
    q.init(a.space, a.boxes + 6 * (int64_t)i);
    const int32_t m = find_ordered(
        s_item, a.ninner,
        [&](uint32_t node, bool& in_l, bool& in_r, uint32_t& lc, uint32_t& rc) {
          float gl, gr;
          find_visit<true, 3>(a.fnodes, node, q, gl, gr, lc, rc);
          in_l = !(gl > 0.0f);
          in_r = !(gr > 0.0f);
        },
        [&](int32_t pos) {
          const int32_t j = a.leaf_ids[pos];
          return j > i && (int64_t)j < a.n && isect_test(a, i, j, pos);
        },
        [&](int32_t k, int32_t pos) {
          if (k >= c) return;
          a.first[(int64_t)a.step * (o + k)] = i;
          a.second[(int64_t)a.step * (o + k)] = a.leaf_ids[pos];
        });
    if (m < 0 && threadIdx.x == 0) atomicOr(a.status, 1);
  }
}

// The same a lane per triangle, where the compact nodes cannot serve.
__global__ __launch_bounds__(kBlock) void k_isect_more_lane(IsectArgs a) {
  __shared__ int32_t s_stack[stack_lds_words(kBlock)];
  const uint32_t n = *a.nmore;
  for (uint32_t e = blockIdx.x * blockDim.x + threadIdx.x; e < n; e += gridDim.x * blockDim.x) {
    const int64_t i = a.more[e];
    const int32_t o = a.poff[i], c = a.npair[i];
    int32_t m = 0;
    isect_walk(a, i, lane_stack_base(s_stack), [&](int32_t j, int32_t) {
      if (m < c) {
        a.first[(int64_t)a.step * (o + m)] = (int32_t)i;
        a.second[(int64_t)a.step * (o + m)] = j;
      }
      ++m;
    });
  }
}

__global__ __launch_bounds__(kBlock) void k_flag_emit(const int32_t* __restrict__ flag,
                                                      const int32_t* __restrict__ off, int64_t n,
                                                      int32_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && flag[i]) out[off[i]] = (int32_t)i;
}

// Batched primal::intersect(Triangle3, Triangle3, includeBoundary, EPS).
__global__ __launch_bounds__(kBlock) void k_tri_tri(const double* __restrict__ t1,
                                                    const double* __restrict__ t2, int64_t n,
                                                    bool inc, double eps,
                                                    uint8_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double* a = t1 + 9 * i;
  const double* b = t2 + 9 * i;
  out[i] = tri_tri_intersect(load_v3(a), load_v3(a + 3), load_v3(a + 6), load_v3(b), load_v3(b + 3),
                             load_v3(b + 6), inc, eps)
               ? 1
               : 0;
}

// Bounding box of each cell of `npc` nodes (primal::compute_bounding_box of
// the cell's points: BoundingBox::addPoint of each, BoundingBox.hpp:466-482,
// a coordinate replaces the bound it is strictly below / above). A node index
// outside [0, nverts) sets bit 1 of *status.
__global__ __launch_bounds__(kBlock) void k_cell_boxes_n(const double* __restrict__ x,
                                                         const double* __restrict__ y,
                                                         const double* __restrict__ z,
                                                         int64_t nverts,
                                                         const int32_t* __restrict__ conn,
                                                         int64_t ncells, int npc,
                                                         double* __restrict__ boxes,
                                                         int32_t* __restrict__ status) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncells) return;
  double b[6] = {kDblMax, kDblMax, kDblMax, -kDblMax, -kDblMax, -kDblMax};
  for (int k = 0; k < npc; ++k) {
    const int32_t v = conn[c * npc + k];
    if (v < 0 || (int64_t)v >= nverts) {
      atomicOr(status, 1);
      continue;
    }
    const double p[3] = {x[v], y[v], z[v]};
    for (int d = 0; d < 3; ++d) {
      if (p[d] < b[d]) b[d] = p[d];
      if (p[d] > b[3 + d]) b[3 + d] = p[d];
    }
  }
  double* o = boxes + 6 * c;
  for (int k = 0; k < 6; ++k) o[k] = b[k];
}

// The first member of every candidate pair: query cell i at
// [offsets[i], offsets[i] + counts[i]).
__global__ __launch_bounds__(kBlock) void k_expand_first(const int32_t* __restrict__ offsets,
                                                         const int32_t* __restrict__ counts,
                                                         int64_t nq, int32_t* __restrict__ first) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nq) return;
  const int32_t o = offsets[i], c = counts[i];
  for (int32_t j = 0; j < c; ++j) first[o + j] = (int32_t)i;
}

// Device allocations of one call, freed on every exit path.
struct Scratch {
  std::vector<void*> ptrs;
  axsq_alloc_fn fn = nullptr;  // the caller's, whose blocks stay its own
  void* ctx = nullptr;
  template <class T>
  int alloc(T** p, int64_t count) {
    *p = nullptr;
    const size_t bytes = sizeof(T) * (size_t)(count > 0 ? count : 1);
    if (fn) {
      *p = static_cast<T*>(fn(ctx, (int64_t)bytes));
      if (*p) return AXSQ_OK;
      set_error("the caller's allocator gave no %zu bytes", bytes);
      return AXSQ_ERR_NOMEM;
    }
    if (hipMalloc((void**)p, bytes) != hipSuccess) {
      *p = nullptr;
      set_error("device allocation of %zu bytes failed", bytes);
      return AXSQ_ERR_NOMEM;
    }
    ptrs.push_back(*p);
    return AXSQ_OK;
  }
  void keep(void* p) {  // ownership passes to the caller
    for (auto& q : ptrs)
      if (q == p) q = nullptr;
  }
  ~Scratch() {
    for (void* p : ptrs)
      if (p) (void)hipFree(p);
  }
};

}  // namespace
}  // namespace axsq

using namespace axsq;

extern "C" int axsq_tri_tri_intersect(const double* t1, const double* t2, int64_t n,
                                      int include_boundary, double eps, uint8_t* out,
                                      void* stream) {
  clear_error();
  if (n < 0 || (n > 0 && (!t1 || !t2 || !out))) {
    set_error("axsq_tri_tri_intersect: need n >= 0 and non-NULL arrays");
    return AXSQ_ERR_INVALID_ARG;
  }
  if (n == 0) return AXSQ_OK;
  hipStream_t s = (hipStream_t)stream;
  k_tri_tri<<<grid_for(n), kBlock, 0, s>>>(t1, t2, n, include_boundary != 0, eps, out);
  AXSQ_CHECK_HIP(hipGetLastError());
  AXSQ_CHECK_HIP(hipStreamSynchronize(s));
  return AXSQ_OK;
}

namespace {
// first / second: an array each; pairs: one array of (first, second) records
// and `degenerate`, from the caller's allocator.
int self_intersections(const double* x, const double* y, const double* z, int64_t nverts,
                       const int32_t* tris, int64_t ntris, double threshold, int32_t** first,
                       int32_t** second, int32_t** pairs, int64_t* npairs, int32_t** degenerate,
                       int64_t* ndegen, axsq_alloc_fn alloc, void* ctx, void* stream) {
  clear_error();
  if (!((first && second) || pairs) || !npairs || !degenerate || !ndegen) {
    set_error("axsq_mesh_self_intersections: NULL output");
    return AXSQ_ERR_INVALID_ARG;
  }
  if (pairs)
    *pairs = nullptr;
  else
    *first = *second = nullptr;
  *degenerate = nullptr;
  *npairs = *ndegen = 0;
  if (ntris < 0 || nverts < 0 || ntris > 0x3fffffffll || nverts > 0x7fffffffll ||
      (ntris > 0 && (!x || !y || !z || !tris || nverts < 1))) {
    set_error("axsq_mesh_self_intersections: invalid mesh arguments");
    return AXSQ_ERR_INVALID_ARG;
  }
  hipStream_t s = (hipStream_t)stream;
  Scratch out;  // the caller's arrays until they are handed over
  out.fn = alloc;
  out.ctx = ctx;
  int32_t *pf = nullptr, *ps = nullptr, *pd = nullptr;
  // pairs: the second member of a record after the first
  auto alloc_out = [&](int64_t np, int64_t nd) -> int {
    AXSQ_TRY(out.alloc(&pf, pairs ? 2 * np : np));
    if (pairs)
      ps = pf + 1;
    else
      AXSQ_TRY(out.alloc(&ps, np));
    return out.alloc(&pd, nd);
  };
  if (ntris == 0) {
    AXSQ_TRY(alloc_out(0, 0));
  } else {
    const int64_t n = ntris;
    Workspace& ws = workspace();
    // records of the vertices where the three arrays outgrow the L2s: crossing noisy
    // spheres of 163,842 / 327,684 / 655,362 / 1,310,724 vertices, a call with them 517 /
    // 728 / 1130 / 2016 us, without 508 / 717 / 1158 / 2076
    const bool pack = nverts >= 524288;
    AXSQ_TRY(ws.mesh_tri.ensure(sizeof(TriRec) * n + (pack ? 32 * (size_t)nverts : 0)));
    AXSQ_TRY(ws.mesh_box.ensure(sizeof(double) * 6 * n));
    AXSQ_TRY(ws.mesh_int.ensure(sizeof(int32_t) * (5 * n + 2) + 2 * sizeof(int64_t) + 64));
    AXSQ_TRY(ws.mesh_slots.ensure(sizeof(int32_t) * kPairSlots * n));
    TriRec* tri = ws.mesh_tri.as<TriRec>();
    double2* verts = pack ? reinterpret_cast<double2*>(tri + n) : nullptr;
    double* boxes = ws.mesh_box.as<double>();
    int64_t* tot = reinterpret_cast<int64_t*>(ws.mesh_int.as<char>());
    int32_t* degf = reinterpret_cast<int32_t*>(tot + 2);
    int32_t* degoff = degf + n;
    int32_t* npair = degoff + n;
    int32_t* poff = npair + n;
    int32_t* more = poff + n;
    int32_t* status = more + n;  // and the length of `more`
    AXSQ_TRY(fill_i32(status, 0, 2, s));
    {
      ProfRange pr("mesh_isect_setup", s);
      if (pack) {
        k_pack_verts<<<grid_for(nverts), kBlock, 0, s>>>(x, y, z, nverts, verts);
        AXSQ_CHECK_HIP(hipGetLastError());
      }
      k_tri_setup<<<grid_for(n), kBlock, 0, s>>>(x, y, z, verts, tris, n, nverts, tri, boxes, degf,
                                                 npair, status);
      AXSQ_CHECK_HIP(hipGetLastError());
    }
    // the BVH over the corner boxes, default scale (MeshTester_detail.hpp:322-338)
    if (!ws.mesh_bvh) {
      ws.mesh_bvh = new axsq_bvh();
      hipGetDevice(&ws.mesh_bvh->device);
    }
    const int rc = bvh_build_into(ws.mesh_bvh, boxes, n, 1.000123, AXSQ_FP64, s);
    if (rc != AXSQ_OK) {
      axsq_bvh_destroy(ws.mesh_bvh);
      ws.mesh_bvh = nullptr;
      return rc;
    }
    const axsq_bvh* b = ws.mesh_bvh;
    IsectArgs a;
    a.nodes = b->nodes;
    a.ninner = (int32_t)(b->n - 1);
    a.fnodes = b->fnodes;
    a.leaf_ids = b->leaf_ids;
    a.leaf_boxes = b->leaf_boxes;
    a.tri = tri;
    a.boxes = boxes;
    a.n = n;
    a.eps = threshold;
    a.npair = npair;
    a.slots = ws.mesh_slots.as<int32_t>();
    a.poff = poff;
    a.more = more;
    a.nmore = reinterpret_cast<uint32_t*>(status + 1);
    a.status = b->status;
    const bool compact = b->find_ok && find_space(b->bounds, a.space);
    {
      ProfRange pr("mesh_isect_walk", s);
      if (compact) {
        // fewer triangles a wave where there are few, to fill the chip
        int tris = 8;
        while (tris < kPoolTris && n > (int64_t)tris * 4096) tris *= 2;
        k_isect_pool<<<(unsigned)((n + tris - 1) / tris), kWaveLanes, 0, s>>>(a, tris);
      } else {
        k_isect_count<<<grid_for(n), kBlock, 0, s>>>(a);
      }
      AXSQ_CHECK_HIP(hipGetLastError());
    }
    AXSQ_TRY(scan_exclusive_i32(npair, poff, n, tot, ws, s));
    AXSQ_TRY(scan_exclusive_i32(degf, degoff, n, tot + 1, ws, s));
    ReadBack r;
    r.total[0] = tot;
    r.total[1] = tot + 1;
    r.status[0] = b->status;
    r.status[1] = status;
    ReadValues v;
    AXSQ_TRY(read_back(r, &v, s));
    if (v.status[1]) {
      set_error("axsq_mesh_self_intersections: connectivity refers to a vertex outside [0, %lld)",
                (long long)nverts);
      return AXSQ_ERR_INVALID_ARG;
    }
    AXSQ_TRY(status_error(v.status[0]));
    const int64_t* totals = v.total;
    AXSQ_TRY(alloc_out(totals[0], totals[1]));
    a.step = pairs ? 2 : 1;
    a.first = pf;
    a.second = ps;
    {
      ProfRange pr("mesh_isect_emit", s);
      k_isect_emit<<<grid_for(n), kBlock, 0, s>>>(a);
      AXSQ_CHECK_HIP(hipGetLastError());
      if (compact)
        k_isect_more<<<(unsigned)std::min<int64_t>(n, 8192), kWaveLanes, 0, s>>>(a);
      else
        k_isect_more_lane<<<std::min(grid_for(n), 1024u), kBlock, 0, s>>>(a);
      AXSQ_CHECK_HIP(hipGetLastError());
      k_flag_emit<<<grid_for(n), kBlock, 0, s>>>(degf, degoff, n, pd);
      AXSQ_CHECK_HIP(hipGetLastError());
    }
    AXSQ_CHECK_HIP(hipStreamSynchronize(s));
    prof_flush();
    *npairs = totals[0];
    *ndegen = totals[1];
  }
  out.keep(pf);
  out.keep(ps);
  out.keep(pd);
  if (pairs) {
    *pairs = pf;
  } else {
    *first = pf;
    *second = ps;
  }
  *degenerate = pd;
  return AXSQ_OK;
}

// As above: first / second or pairs.
int mesh_candidates(const double* ix, const double* iy, const double* iz, int64_t inverts,
                    const int32_t* icells, int64_t nicells, const double* qx, const double* qy,
                    const double* qz, int64_t qnverts, const int32_t* qcells, int64_t nqcells,
                    int nodes_per_cell, int32_t** first, int32_t** second, int32_t** pairs,
                    int64_t* npairs, axsq_alloc_fn alloc, void* ctx, void* stream) {
  clear_error();
  if (!((first && second) || pairs) || !npairs) {
    set_error("axsq_mesh_candidates: NULL output");
    return AXSQ_ERR_INVALID_ARG;
  }
  if (pairs)
    *pairs = nullptr;
  else
    *first = *second = nullptr;
  *npairs = 0;
  if (nodes_per_cell < 1 || nodes_per_cell > 8) {
    set_error("axsq_mesh_candidates: nodes_per_cell %d outside [1, 8]", nodes_per_cell);
    return AXSQ_ERR_INVALID_ARG;
  }
  if (nicells < 0 || nqcells < 0 || nicells > 0x3fffffffll || nqcells > 0x3fffffffll ||
      inverts < 0 || qnverts < 0 || inverts > 0x7fffffffll || qnverts > 0x7fffffffll ||
      (nicells > 0 && (!ix || !iy || !iz || !icells)) ||
      (nqcells > 0 && (!qx || !qy || !qz || !qcells))) {
    set_error("axsq_mesh_candidates: invalid mesh arguments");
    return AXSQ_ERR_INVALID_ARG;
  }
  hipStream_t s = (hipStream_t)stream;
  Scratch out;
  out.fn = alloc;
  out.ctx = ctx;
  int32_t *pf = nullptr, *ps = nullptr;  // pairs: pf alone, of records
  int64_t total = 0;
  if (nicells == 0 || nqcells == 0) {
    AXSQ_TRY(out.alloc(&pf, 0));
    if (!pairs) AXSQ_TRY(out.alloc(&ps, 0));
  } else {
    const int64_t ni = nicells, nq = nqcells;
    Workspace& ws = workspace();
    AXSQ_TRY(ws.mesh_box.ensure(sizeof(double) * 6 * ni));
    AXSQ_TRY(ws.mesh_tri.ensure(sizeof(double) * 6 * nq));
    // mesh_int: totals (2 x int64), status, then offsets and counts
    AXSQ_TRY(ws.mesh_int.ensure(2 * sizeof(int64_t) + sizeof(int32_t) * (2 * nq + 2)));
    double* ibox = ws.mesh_box.as<double>();
    double* qbox = ws.mesh_tri.as<double>();
    int64_t* tot = reinterpret_cast<int64_t*>(ws.mesh_int.as<char>());
    int32_t* status = reinterpret_cast<int32_t*>(tot + 2);
    int32_t* offsets = status + 2;
    int32_t* counts = offsets + nq;
    AXSQ_TRY(fill_i32(status, 0, 1, s));
    k_cell_boxes_n<<<grid_for(ni), kBlock, 0, s>>>(ix, iy, iz, inverts, icells, ni,
                                                   nodes_per_cell, ibox, status);
    AXSQ_CHECK_HIP(hipGetLastError());
    k_cell_boxes_n<<<grid_for(nq), kBlock, 0, s>>>(qx, qy, qz, qnverts, qcells, nq,
                                                   nodes_per_cell, qbox, status);
    AXSQ_CHECK_HIP(hipGetLastError());
    // the BVH over the insert mesh's boxes, default scale
    // (quest_candidates_example.cpp:420-423)
    if (!ws.mesh_bvh) {
      ws.mesh_bvh = new axsq_bvh();
      hipGetDevice(&ws.mesh_bvh->device);
    }
    const int rc = bvh_build_into(ws.mesh_bvh, ibox, ni, 1.000123, AXSQ_FP64, s);
    if (rc != AXSQ_OK) {
      axsq_bvh_destroy(ws.mesh_bvh);
      ws.mesh_bvh = nullptr;
      return rc;
    }
    const axsq_bvh* b = ws.mesh_bvh;
    // findBoundingBoxes for every query box (:426-434): one walk, the first
    // ids kept, the rest walked again
    const int kstash = stash_slots(nq);
    AXSQ_TRY(ws.find_stash.ensure(sizeof(int32_t) * kstash * (size_t)nq));
    AXSQ_TRY(ws.find_cnt.ensure(sizeof(int32_t) * (size_t)nq));
    AXSQ_TRY(ws.find_over.ensure(sizeof(int32_t) * (size_t)nq));
    if (!ws.find_n.p) ws.find_n_zero = false;
    AXSQ_TRY(ws.find_n.ensure(sizeof(int64_t) * 2));  // the list's length as in find_count_impl
    uint32_t* nover = reinterpret_cast<uint32_t*>(ws.find_n.as<int64_t>() + 1);
    if (!ws.find_n_zero) AXSQ_TRY(fill_i32(reinterpret_cast<int32_t*>(nover), 0, 1, s));
    ws.find_n_zero = false;
    const double tol = 2.220446049250313e-16;  // BVH default tolerance (unused by boxes)
    AXSQ_TRY(find_launch(b, AXSQ_QUERY_BOXES, 0, qbox, nullptr, nullptr, 6, nq, tol, counts,
                         nullptr, nullptr, nullptr, ws.find_stash.as<int32_t>(), kstash,
                         ws.find_cnt.as<int32_t>(), ws.find_over.as<int32_t>(), nover, s));
    AXSQ_TRY(scan_exclusive_i32(counts, offsets, nq, tot, ws, s));
    ReadBack r;
    r.total[0] = tot;
    r.list = nover;
    r.nlist = 1;
    r.status[0] = b->status;
    r.status[1] = status;
    ReadValues v;
    AXSQ_TRY(read_back(r, &v, s));
    ws.find_n_zero = true;
    if (v.status[1]) {
      set_error("axsq_mesh_candidates: a cell refers to a vertex outside its mesh");
      return AXSQ_ERR_INVALID_ARG;
    }
    AXSQ_TRY(status_error(v.status[0]));
    total = v.total[0];
    if (total > 0x7fffffffll) {
      set_error("axsq_mesh_candidates: %lld candidate pairs exceed the int32 index range",
                (long long)total);
      return AXSQ_ERR_INVALID_ARG;
    }
    AXSQ_TRY(out.alloc(&pf, pairs ? 2 * total : total));
    if (!pairs) AXSQ_TRY(out.alloc(&ps, total));
    // the pair list (:440-458): query cell, then its candidates in order
    int32_t* const ids = pairs ? pf : ps;
    AXSQ_TRY(stash_copy_launch(b, AXSQ_QUERY_BOXES, pairs != nullptr,
                               ws.find_stash.as<int32_t>(), kstash, ws.find_cnt.as<int32_t>(),
                               offsets, nq, ids, s));
    if (v.list > 0)
      AXSQ_TRY(find_launch(b, AXSQ_QUERY_BOXES, 2, qbox, nullptr, nullptr, 6, v.list, tol,
                           nullptr, counts, offsets, ids, nullptr, 0, nullptr,
                           ws.find_over.as<int32_t>(), nullptr, s, pairs != nullptr));
    if (!pairs) {
      k_expand_first<<<grid_for(nq), kBlock, 0, s>>>(offsets, counts, nq, pf);
      AXSQ_CHECK_HIP(hipGetLastError());
    }
    AXSQ_CHECK_HIP(hipStreamSynchronize(s));
    prof_flush();
  }
  out.keep(pf);
  out.keep(ps);
  if (pairs) {
    *pairs = pf;
  } else {
    *first = pf;
    *second = ps;
  }
  *npairs = total;
  return AXSQ_OK;
}
}  // namespace

extern "C" int axsq_mesh_self_intersections(const double* x, const double* y, const double* z,
                                            int64_t nverts, const int32_t* tris, int64_t ntris,
                                            double threshold, int32_t** first, int32_t** second,
                                            int64_t* npairs, int32_t** degenerate,
                                            int64_t* ndegen, void* stream) {
  return self_intersections(x, y, z, nverts, tris, ntris, threshold, first, second, nullptr,
                            npairs, degenerate, ndegen, nullptr, nullptr, stream);
}

extern "C" int axsq_mesh_self_intersections_alloc(const double* x, const double* y,
                                                  const double* z, int64_t nverts,
                                                  const int32_t* tris, int64_t ntris,
                                                  double threshold, axsq_alloc_fn alloc,
                                                  void* ctx, int32_t** pairs, int64_t* npairs,
                                                  int32_t** degenerate, int64_t* ndegen,
                                                  void* stream) {
  if (!alloc || !pairs) {
    set_error("axsq_mesh_self_intersections_alloc: NULL allocator or output");
    return AXSQ_ERR_INVALID_ARG;
  }
  return self_intersections(x, y, z, nverts, tris, ntris, threshold, nullptr, nullptr, pairs,
                            npairs, degenerate, ndegen, alloc, ctx, stream);
}

extern "C" int axsq_mesh_candidates(const double* ix, const double* iy, const double* iz,
                                    int64_t inverts, const int32_t* icells, int64_t nicells,
                                    const double* qx, const double* qy, const double* qz,
                                    int64_t qnverts, const int32_t* qcells, int64_t nqcells,
                                    int nodes_per_cell, int32_t** first, int32_t** second,
                                    int64_t* npairs, void* stream) {
  return mesh_candidates(ix, iy, iz, inverts, icells, nicells, qx, qy, qz, qnverts, qcells,
                         nqcells, nodes_per_cell, first, second, nullptr, npairs, nullptr,
                         nullptr, stream);
}

extern "C" int axsq_mesh_candidates_alloc(const double* ix, const double* iy, const double* iz,
                                          int64_t inverts, const int32_t* icells,
                                          int64_t nicells, const double* qx, const double* qy,
                                          const double* qz, int64_t qnverts,
                                          const int32_t* qcells, int64_t nqcells,
                                          int nodes_per_cell, axsq_alloc_fn alloc, void* ctx,
                                          int32_t** pairs, int64_t* npairs, void* stream) {
  if (!alloc || !pairs) {
    set_error("axsq_mesh_candidates_alloc: NULL allocator or output");
    return AXSQ_ERR_INVALID_ARG;
  }
  return mesh_candidates(ix, iy, iz, inverts, icells, nicells, qx, qy, qz, qnverts, qcells,
                         nqcells, nodes_per_cell, nullptr, nullptr, pairs, npairs, alloc, ctx,
                         stream);
}
