// Device BVH builder: Morton-ordered primitives, level-synchronous binned SAH
// splits, collapse to 4-wide nodes; and the traversal's 8-wide nodes from the
// 4-wide tree of either builder.
#pragma once

#include <cstdint>

#include "scene_host.h"

namespace rad {

struct DeviceBvhStats {
  uint32_t node_count = 0;  // 4-wide nodes
  uint32_t depth = 0;       // 4-wide levels
  uint32_t stack_need = 0;  // traversal stack entries the tree can need (kTraceStackEntries)
  uint32_t levels = 0;      // binary build levels
  float sah_cost = 0;
  double build_ms = 0;
};

// Consecutive primitives [begin, next segment's begin) of one shape, in shape
// order: the triangles of a mesh from tri_offset on, or the one primitive of
// another shape (other: its index in PrimSource::other_rec; 0xffffffff for a
// mesh).
struct PrimSegment {
  uint32_t begin, geom, tri_offset, other;
};

// Where a scene's primitives come from: triangles are in device memory already
// (DevScene::tris), the few others come from the host (three float4 and six
// floats of bounds each).
struct PrimSource {
  std::vector<PrimSegment> segs;
  std::vector<float4> other_rec;
  std::vector<float> other_box;
  const float4* d_tris = nullptr;
  uint32_t count = 0;
};

// Writes the nodes and the primitive records in leaf order to device buffers,
// whose old contents hold until outputsValid is cleared, just before the first
// write; work: scratch memory, left allocated for BuildWideNodes.
void BuildBvh4Device(const PrimSource& src, int maxLeaf, hipStream_t st, DeviceBuffer& nodesOut, DeviceBuffer& primsOut,
                     bool& outputsValid, DeviceBuffer& work, DeviceBvhStats& stats);

// The traversal's nodes from a tree of m BvhNode4, with leaves of at most
// maxLeaf, over n primitive records (device buffers): writes them to `out` and
// returns their number, puts the primitive records in the order of their leaves
// and renumbers the BvhNode4 leaves to match; throws if a child box cannot be
// bounded.  work: scratch memory, reused when large enough.
uint32_t BuildWideNodes(DeviceBuffer& nodes, uint32_t m, uint32_t maxLeaf, DeviceBuffer& prims, uint32_t n, hipStream_t st,
                        DeviceBuffer& work, DeviceBuffer& out);

}  // namespace rad
