// Host side of the tree builds, for tests/test_bvh_host.py: one translation
// unit with the host builder and the 8-wide nodes, compiled without a device.
#include "bvh_build.cpp"
#include "bvh_wide.h"

using namespace rad;

extern "C" uint32_t probe_host_leaf(const float* bounds, uint32_t n, int max_leaf, uint32_t* stack_need) {
  BvhBuildResult r;
  BuildBvh4Host(bounds, n, max_leaf, r);
  *stack_need = r.stack_need;
  return BvhLargestLeaf(r.nodes);
}
extern "C" uint32_t probe_max_leaf_prims() { return kMaxLeafPrims; }

// The 8-wide nodes of a BvhNode4 tree over the primitives `order`.  Returns
// the errors found: CheckWideNodes, primitives not placed exactly once,
// BvhNode4 leaves that do not name their primitives' new places.  out: nodes,
// the traversal's stack need, the BvhNode4 tree's.
static uint32_t Wide(std::vector<BvhNode4>& nodes, const float* bounds, const std::vector<uint32_t>& order, uint32_t out[3],
                     std::vector<BvhNode8>& wide, std::vector<float>& boxes) {
  const uint32_t n = uint32_t(order.size());
  const std::vector<BvhNode4> before = nodes;
  std::vector<uint32_t> perm, seen(n, 0);
  uint32_t errors = 0;
  BuildWideNodesHost(nodes, n, wide, perm);
  boxes.clear();
  for (uint32_t p : perm) {
    if (p >= n || seen[p]++) return 1;
    boxes.insert(boxes.end(), bounds + 6 * size_t(order[p]), bounds + 6 * size_t(order[p]) + 6);
  }
  for (size_t x = 0; x < nodes.size(); x++)
    for (int s = 0; s < 4; s++)
      for (uint32_t q = 0; q < nodes[x].count[s]; q++) errors += perm[nodes[x].child[s] + q] != before[x].child[s] + q;
  out[0] = uint32_t(wide.size());
  out[2] = BvhStackNeed(nodes);
  return errors + CheckWideNodes(wide, boxes.data(), n, &out[1]);
}

extern "C" uint32_t probe_wide_host(const float* bounds, uint32_t n, int max_leaf, uint32_t out[3]) {
  BvhBuildResult r;
  BuildBvh4Host(bounds, n, max_leaf, r);
  std::vector<BvhNode8> wide;
  std::vector<float> boxes;
  return Wide(r.nodes, bounds, r.order, out, wide, boxes);
}

// CheckWideNodes of a host-built tree in which one thing of node x is wrong:
// what 0-5 a plane (lo / hi of x, y, z) of child slot s is moved inside its
// box, 6 its primitives and 7 its inner children are the next ones.  -1: the
// node has no such thing.
extern "C" int32_t probe_wide_broken(const float* bounds, uint32_t n, uint32_t x, int s, int what) {
  BvhBuildResult r;
  BuildBvh4Host(bounds, n, 4, r);
  std::vector<BvhNode8> wide;
  std::vector<float> boxes;
  uint32_t out[3];
  if (Wide(r.nodes, bounds, r.order, out, wide, boxes)) return -2;
  x %= uint32_t(wide.size());
  BvhNode8& w = wide[x];
  uint16_t* plane[6] = {w.lox, w.hix, w.loy, w.hiy, w.loz, w.hiz};
  if (what < 6) {
    const uint32_t lo = plane_value(plane[what & ~1][s]), hi = plane_value(plane[what | 1][s]);
    if (lo >= hi) return -1;  // an empty slot
    plane[what][s] = plane_bits(what & 1 ? lo : hi);
  } else if (what == 6) {
    if ((w.ends[1] >> 24) == 0) return -1;
    w.prim_base++;
  } else {
    if (!(w.exps >> 24)) return -1;
    w.child_base++;
  }
  return int32_t(CheckWideNodes(wide, boxes.data(), n));
}

// A chain of `length` BvhNode4 with `inner` inner children (the others end in
// one leaf) and leaves of the given sizes, primitive i at x = i.
extern "C" uint32_t probe_wide_chain(uint32_t length, uint32_t inner, const uint32_t* leaves, uint32_t nLeaves, uint32_t out[3]) {
  std::vector<BvhNode4> nodes;
  std::vector<float> bounds;
  std::vector<uint32_t> order;
  auto leaf = [&](BvhNode4& nd, int s, uint32_t c) {
    nd.child[s] = int32_t(order.size());
    nd.count[s] = c;
    nd.lox[s] = float(order.size()), nd.hix[s] = float(order.size() + c);
    nd.loy[s] = nd.loz[s] = 0.f, nd.hiy[s] = nd.hiz[s] = 1.f;
    for (uint32_t i = 0; i < c; i++) {
      const float x = float(order.size());
      bounds.insert(bounds.end(), {x, 0.f, 0.f, x + 1.f, 1.f, 1.f});
      order.push_back(uint32_t(order.size()));
    }
  };
  auto blank = [] {
    BvhNode4 nd{};
    for (int s = 0; s < 4; s++) nd.child[s] = -1, nd.lox[s] = nd.loy[s] = nd.loz[s] = kInf, nd.hix[s] = nd.hiy[s] = nd.hiz[s] = -kInf;
    return nd;
  };
  std::vector<std::pair<uint32_t, int>> links;  // (node, slot) that the next node of the chain hangs from
  for (uint32_t l = 0; l < length; l++) {
    const uint32_t x = uint32_t(nodes.size());
    nodes.push_back(blank());
    for (uint32_t k = 0; k < nLeaves; k++) leaf(nodes[x], int(k), leaves[k]);
    for (uint32_t k = 0; k + 1 < inner; k++) {  // side branches: one node with one leaf
      const uint32_t y = uint32_t(nodes.size());
      nodes.push_back(blank());
      leaf(nodes[y], 0, 1);
      BvhNode4& nd = nodes[x];
      const int s = int(nLeaves + k);
      nd.child[s] = int32_t(y), nd.count[s] = 0;
      nd.lox[s] = nodes[y].lox[0], nd.hix[s] = nodes[y].hix[0], nd.loy[s] = nd.loz[s] = 0.f, nd.hiy[s] = nd.hiz[s] = 1.f;
    }
    if (l + 1 < length && inner) links.push_back({x, int(nLeaves + inner - 1)});
  }
  for (const auto& [x, s] : links) {
    nodes[x].child[s] = int32_t(x + inner);  // each link adds itself and inner - 1 side branches
    nodes[x].count[s] = 0;
    nodes[x].lox[s] = nodes[x].loy[s] = nodes[x].loz[s] = 0.f;
    nodes[x].hix[s] = float(order.size()), nodes[x].hiy[s] = nodes[x].hiz[s] = 1.f;
  }
  for (BvhNode4& nd : nodes)
    for (int s = 0; s < 4; s++) {
      if (nd.child[s] < 0) continue;
      nd.lox[s] = Widen(nd.lox[s], false), nd.loy[s] = Widen(nd.loy[s], false), nd.loz[s] = Widen(nd.loz[s], false);
      nd.hix[s] = Widen(nd.hix[s], true), nd.hiy[s] = Widen(nd.hiy[s], true), nd.hiz[s] = Widen(nd.hiz[s], true);
    }
  std::vector<BvhNode8> wide;
  std::vector<float> boxes;
  return Wide(nodes, bounds.data(), order, out, wide, boxes);
}
