// Host-side octree (the reference's Octree<Renderable<BakedTriFace>> after
// push + build) and its flattening into the device traversal layout.
#pragma once
#include <vector>
#include "dr_geom.h"

namespace dr {

constexpr int kMaxTreeDepth = 24;          // OCTREE_MAX_DEPTH (Octree.cuh:13); traversal stack bound

struct OctreeHost {
  int split_threshold = 8, max_depth = 24;
  std::vector<Tri> tris;                   // push order = hit id
  // nodes in breadth-first order; the 8 children of a node are contiguous
  std::vector<Box> bounds;
  std::vector<int32_t> children;           // first child, -1 = leaf
  std::vector<int32_t> list_off, list;     // leaf triangle lists (stored order)
};

// Builds the octree over tris9 (ntris x 9 floats).  nthreads <= 0: all cores.
// Returns 0, -1 for bad arguments, -2 if the node pool overflowed.
int build_octree(const float *tris9, int ntris, int split_threshold, int max_depth, int nthreads, OctreeHost &out);

// ---------------------------------------------------------------- device layout
// A "group" is the 8 contiguous children of one interior node: 32 words, one 128-B line.
//   [0..2]   origin of the group's grid          [3]  head (below)
//   [4..6]   cell size of the grid per axis      [7]  group of the first interior child
//   [8..19]  child boxes in grid cells, one byte each: min.x[8] min.y[8] min.z[8] max.x[8]
//            max.y[8] max.z[8]
//   [20..28] first leaf entry of child k, and the end of child 7's (child k holds the entries
//            [20 + k] .. [21 + k]; none if it is interior or empty)
//   head: bits 0-7: child k has a non-empty leaf at or below it; bits 8-15: child k is interior
// Interior children get consecutive groups (breadth-first order), so interior child k's group is
// word 7 plus the number of interior children before k.
// Child k uses the reference's numbering (bit0 = z-high, bit1 = y-high, bit2 = x-high).
// A child's grid box holds every non-empty leaf box at or below it (rounded outwards, checked in
// double when flattening), so it decides only which subtrees can be skipped.  The reference's own
// decisions, the slab tests of the leaf and of its ancestors, are taken from the node records
// when a hit is about to be accepted.
constexpr int kGroupWords = 32;
constexpr int kGroupF4 = kGroupWords / 4;
constexpr int kGroupHead = 3, kGroupBase = 7, kGroupBoxes = 8, kGroupEntry = 20;
// A node record, 8 words: min.x min.y min.z max.x | max.y max.z parent nested.  Node 8 * g + k is
// child k of group g; parent is the parent's node, -1 under the root; nested is 1 if the box lies
// inside the box of every ancestor, the root included.
constexpr int kNodeWords = 8, kNodeF4 = kNodeWords / 4;
// A triangle record is 16 words (64 B):
//   a.x a.y a.z n.x | n.y n.z b.x b.y | b.z c.x c.y c.z | thr0 thr1 thr2 id
// n = (b-a) x (c-a) and thr* = the ray-independent right-hand sides of the
// containsVertex test; the plane test reads only the first 32 B.
// Degenerate triangles (always a miss) get no record.  Records exist in two layouts:
// one per leaf entry in leaf order (read by the render kernels) and one per distinct
// triangle with a leaf-entry -> record index (read by the closest-hit kernel, whose
// random rays touch the whole scene: the compact layout fits the last-level cache).
constexpr int kRecWords = 16;

struct OctreeFlat {
  std::vector<float> groups;               // ngroups * kGroupWords words (ints stored bitwise)
  std::vector<float> nodes;                // 8 * ngroups * kNodeWords words
  std::vector<float> recs;                 // nrec * 16 words, one per leaf entry (leaf order)
  std::vector<float> urecs;                // the same records once per distinct triangle
  std::vector<int32_t> lref;               // leaf entry -> its record in urecs
  Box root;
  int root_is_leaf = 0, root_start = 0, root_count = 0;
  int ngroups = 0, nrec = 0;
  int max_depth = 0;                       // depth of the deepest node (root: 0), not the build limit
  double ray_records = 0.0;                // records a random ray through the root box meets: the sum over
                                           // leaves of their records times their box's share of its surface
  float reach = 0.0f;                      // largest magnitude of a box coordinate, inf if one is not finite
};
int flatten_octree(const OctreeHost &t, OctreeFlat &out);

}  // namespace dr
