// Acceleration-structure builders.  Both produce the same 4-wide node layout
// (BvhNode4) over a primitive permutation; the traversal's 8-wide nodes are made
// from it whichever builder ran.  Replaces the Embree BVH build (embree.cpp:18-43).
#pragma once

#include <cstdint>
#include <vector>

#include "scene_dev.h"

namespace rad {

struct BvhBuildResult {
  std::vector<BvhNode4> nodes;
  std::vector<uint32_t> order;  // leaf-order position -> input primitive index
  uint32_t depth = 0;
  uint32_t stack_need = 0;  // traversal stack entries the tree can need (kTraceStackEntries)
  float sah_cost = 0;
  double build_ms = 0;
};

// Host binned-SAH build.  `bounds` holds 6 floats per primitive
// (lo.xyz, hi.xyz).  Leaves hold at most `max_leaf` primitives, but a range
// that is not split apart after 60 levels is one leaf whatever its size.
void BuildBvh4Host(const float* bounds, uint32_t count, int max_leaf, BvhBuildResult& out);

// The traversal's nodes (bvh_wide.h) from a tree over n primitives: their leaf
// order is given as perm (new place -> old place), and the leaves of `nodes` are
// renumbered to match.  Throws if a child box cannot be bounded.
void BuildWideNodesHost(std::vector<BvhNode4>& nodes, uint32_t n, std::vector<BvhNode8>& wide, std::vector<uint32_t>& perm);

// Errors of the traversal's nodes over n primitives (boxes: six floats each, in
// the order of the leaves): primitives not referenced exactly once, node
// references out of range or repeated, child boxes that do not contain the
// primitives below them with half the margin that the builders widen boxes by,
// a stack need (to `need` if given) beyond the traversal's.
uint32_t CheckWideNodes(const std::vector<BvhNode8>& wide, const float* boxes, uint32_t n, uint32_t* need = nullptr);

// SAH cost of a finished tree (traversal 1, intersection 1, relative to root area).
float BvhSahCost(const std::vector<BvhNode4>& nodes);
uint32_t BvhDepth(const std::vector<BvhNode4>& nodes);
// Worst-case traversal stack entries of the tree (see kTraceStackEntries).
uint32_t BvhStackNeed(const std::vector<BvhNode4>& nodes);
// Primitives of the largest leaf.
uint32_t BvhLargestLeaf(const std::vector<BvhNode4>& nodes);

}  // namespace rad
