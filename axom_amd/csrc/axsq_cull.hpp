// axsq_cull.hpp -- oriented child boxes for the signed-distance walk.
//
// The reference walk prunes with axis-aligned boxes. On a slanted patch of
// surface such a box is far thicker than the patch, so a query at distance d
// checks every triangle whose box (not whose surface) comes within d: 154
// triangles and 362 nodes a query on the 81,920-triangle sphere, 765 and
// 1,688 on the 1.3M-triangle one. A second record per inner node holds its
// two children's extents in a frame fitted to the node's surface (mean
// normal, split direction, their cross product). A subtree whose oriented
// box is farther than the running minimum holds no triangle the walk could
// use, and leaving it out leaves 13 triangles and 75 nodes, and 18 and 118.
// Forward and adjoint of 4M queries on the 81,920-triangle sphere: 33.0 ms
// with the reference walk alone, 4.2 ms; a shape-fit iteration on 1.3M
// triangles, 8M queries: 226 and 15.0 ms; 1,000 queries on 5,120 triangles:
// 1.28 and 0.046 ms. Surfaces whose patches are as thick as their boxes gain
// nothing: the build tells them (k_cull_class), and large batches on them take
// the reference walk.
//
// Why the result is the reference walk's, bit for bit. Let s be the running
// minimum (squared) and p the closest point when the reference checks leaf Y.
// The check changes the state only if Y is strictly closer, or if Y's closest
// point lies within 1e-6 of p and adds a pseudo-normal term (checkCandidate,
// SignedDistance.hpp:637-737). Either way Y comes within sqrt(s) + 1e-6 of
// the query.
//  - The walk here visits children in the reference's order and leaves out
//    only subtrees whose every triangle is farther than
//    sqrt(minimum) + 1e-6 + slack, with a minimum no smaller than s. So every
//    leaf that changes the reference's state is checked here, in the same
//    order.
//  - A leaf the reference pruned by its axis-aligned box must not change the
//    state here. A leaf is applied only after its own scaled box passes
//    box distance <= s; if it does not, the query is given to the reference
//    walk. A leaf whose box passes at s is reached by the reference too, since
//    all its tests of that leaf and its ancestors used minima no smaller.
// Leaves that change nothing may be checked by one walk and not by the
// other; the state after each leaf that changes it is the same in both.
//
// Rounding. All of it is in mesh coordinates: x = (q - centre) * scale in
// float, scale a power of two that makes the mesh's diagonal 1 to 2. The
// extents contain every triangle inflated by `tau`, the largest distance its
// computed closest point can have from it (k_cull_leaf), and by the rounding
// of its own projections. A projection is of p = x - m, m the node's middle as
// stored: x is off by 2^-24 |x|, p by 2^-24 |p|, each of three products and
// sums by 2^-24 |p|, so a query's three together by 7.2 2^-24 R (R: its distance
// to the farthest corner of the mesh's box, |x| and |p| at most); the walk's
// slack is 1.2 times that. Frames are orthonormal to 2^-22, covered by a
// relative 2^-18.
// (Projections of x less those of m, off by parts of |x| at every node, took a
// slack of 2^-19 R and 2^-20 about every triangle, more than the tie radius and
// the thickness of a patch of a fine mesh: 4M queries on 2.1M triangles 6.62 ms,
// 6.39 now, 8M on 1.3M (an iteration) 15.7 and 15.2.)
#pragma once

#include "axsq_device.hpp"
#include "axsq_find.hpp"  // halves

namespace axsq {

// Read alone by a visit. The walk's lanes are at different nodes, and the
// vector L1 returns one lane's 16 bytes a cycle: with 128-byte records it was
// busy 96% of the walk's time. So the record is 80 bytes, five loads: two of
// the three axes (the third is their cross product), and the extents as
// halves, rounded outward, relative to m, the middle between the two child
// boxes' centroids. Extents run along w, u, w x u.
// (a, b): the unit vector between those centroids along w and u (it has no
// third component), so a t_w + b t_u > 0, t the projections less m, says
// that the right child is nearer. inv_d: the inverse distance of the
// centroids; a query so near that plane that float rounding could decide
// reads the boxes instead.
struct __attribute__((aligned(16))) CullNode {
  float w[3], u[3];
  float m[3];
  float a, b, inv_d;
  uint32_t l[3], r[3];  // left / right child per axis: halves lo | hi << 16
  int32_t lc, rc;
};
static_assert(sizeof(CullNode) == 80, "CullNode is five 16-byte loads");

// A triangle's part of a pseudo-normal sum: its unit normal and its angle at
// each corner, or -1 where a degenerate triangle adds nothing. Computed once a
// mesh by normal_term's own operations, so the sums are the same: a query on a
// vertex adds about six terms of some 600 FP64 instructions each (square roots,
// divisions, an arc cosine). The walk of 4M queries on 81,920 triangles: 3.77 ms
// without the table, 3.59 with it.
struct __attribute__((aligned(16))) NormRec {
  double un[3];
  double angle[3];
};
static_assert(sizeof(NormRec) == 48, "NormRec is three 16-byte loads");

// Queries farther than this many mesh diagonals from the mesh's farthest
// corner go to the reference walk: tau is computed for that distance.
constexpr double kCullReach = 4.0;

// Mesh coordinates: centre and scale of the mesh's bounding box.
struct CullSpace {
  double o[3];
  double scale;
};

// t: projections of mesh coordinates x less m, by the same operations in the
// build and the walk.
__device__ __forceinline__ void cull_project(const float w[3], const float u[3], const float m[3],
                                             const float x[3], float t[3]) {
  const float v0 = fmaf(w[1], u[2], -(w[2] * u[1]));
  const float v1 = fmaf(w[2], u[0], -(w[0] * u[2]));
  const float v2 = fmaf(w[0], u[1], -(w[1] * u[0]));
  const float p0 = x[0] - m[0], p1 = x[1] - m[1], p2 = x[2] - m[2];
  t[0] = fmaf(p0, w[0], fmaf(p1, w[1], p2 * w[2]));
  t[1] = fmaf(p0, u[0], fmaf(p1, u[1], p2 * u[2]));
  t[2] = fmaf(p0, v0, fmaf(p1, v1, p2 * v2));
}

}  // namespace axsq
