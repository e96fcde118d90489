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
// Forward and adjoint of 4M queries on the 81,920-triangle sphere: 33.2 ms
// with the reference walk alone, 8.7 ms; a shape-fit iteration on 1.3M
// triangles, 8M queries: 226 and 34.8 ms; 1,000 queries on 5,120 triangles:
// 1.8 and 0.08 ms.
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
// Rounding. The extents contain every triangle inflated by `tau`, the
// largest distance its computed closest point can have from it (k_cull_leaf).
// Query coordinates enter as float pairs relative to the node's centre c, so
// a projection is off by at most 2^-21 of |q - c| <= R (R: distance to the
// farthest corner of the mesh's box); the walk's slack covers sqrt(3) times
// that. Frames are orthonormal to 2^-22, covered by a relative 2^-18.
#pragma once

#include "axsq_device.hpp"

namespace axsq {

// 128 bytes, one cache line, beside each Node64: a visit reads this record
// alone. Extents are along w, u, v from c. (dn, dt, inv_d): the plane between
// the two child boxes' centroids, dn the unit vector towards the right one;
// the right child is nearer when dn . (q - c) > dt. inv_d is the inverse
// distance of the centroids: a query so near the plane that float rounding
// could decide reads the boxes instead.
struct __attribute__((aligned(128))) CullNode {
  float c[3];
  float w[3], u[3], v[3];
  float llo[3], lhi[3];
  float rlo[3], rhi[3];
  float dn[3], dt;
  float inv_d;
  int32_t lc, rc;
  int32_t pad;
};
static_assert(sizeof(CullNode) == 128, "CullNode is one cache line");

// Queries farther than this many mesh diagonals from the mesh's farthest
// corner go to the reference walk: tau is computed for that distance.
constexpr double kCullReach = 4.0;

}  // namespace axsq
