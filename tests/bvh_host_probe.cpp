// Host side of the tree builds, for tests/test_bvh_host.py: one translation
// unit with the host builder, compiled without a device.
#include "bvh_build.cpp"

extern "C" uint32_t probe_host_leaf(const float* bounds, uint32_t n, int max_leaf, uint32_t* stack_need) {
  rad::BvhBuildResult r;
  rad::BuildBvh4Host(bounds, n, max_leaf, r);
  *stack_need = r.stack_need;
  return rad::BvhLargestLeaf(r.nodes);
}
extern "C" uint32_t probe_max_leaf_prims() { return rad::kMaxLeafPrims; }
