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

// The 8-wide nodes of a BvhNode4 tree over n primitives.  Returns the errors found: primitives not placed exactly
// once, BvhNode4 leaves that do not name their primitives' new places, wide
// leaves and children that do not lead to every primitive inside the boxes of
// all nodes on the way.  out: nodes, the traversal's stack need, the BvhNode4
// tree's.
static uint32_t Wide(std::vector<BvhNode4>& nodes, const float* bounds, const std::vector<uint32_t>& order, uint32_t out[3]) {
  const uint32_t n = uint32_t(order.size());
  const std::vector<BvhNode4> before = nodes;
  std::vector<BvhNode8> wide;
  std::vector<uint32_t> perm;
  uint32_t errors = 0;
  BuildWideNodesHost(nodes, n, wide, perm);
  std::vector<uint32_t> seen(n, 0), need(wide.size(), 0), reached(n, 0);
  for (uint32_t p : perm)
    if (p >= n || seen[p]++) errors++;
  for (size_t x = 0; x < nodes.size(); x++)
    for (int s = 0; s < 4; s++)
      for (uint32_t q = 0; q < nodes[x].count[s]; q++) errors += perm[nodes[x].child[s] + q] != before[x].child[s] + q;
  struct Box {
    float lo[3], hi[3];
  };
  std::vector<Box> box(wide.size());  // of the primitives below
  for (size_t x = wide.size(); x-- > 0;) {
    const BvhNode8& w = wide[x];
    Box nb{{kInf, kInf, kInf}, {-kInf, -kInf, -kInf}};
    uint32_t inner = 0, begin = 0;
    for (int s = 0; s < 8; s++) {
      const uint32_t end = (w.ends[s >> 2] >> (8 * (s & 3))) & 0xffu;
      Box b{{kInf, kInf, kInf}, {-kInf, -kInf, -kInf}};
      if (w.exps >> 24 >> s & 1u) {
        const uint32_t c = w.child_base + inner++;
        if (c <= x || c >= wide.size()) return errors + 1;
        b = box[c];
        need[x] = std::max(need[x], need[c]);
      } else {
        for (uint32_t k = begin; k < end; k++) {
          if (k >= kWideNodePrims || w.prim_base + k >= n) return errors + 1;
          reached[w.prim_base + k]++;
          const float* p = bounds + 6 * size_t(order[perm[w.prim_base + k]]);
          for (int a = 0; a < 3; a++) b.lo[a] = std::min(b.lo[a], p[a]), b.hi[a] = std::max(b.hi[a], p[3 + a]);
        }
      }
      begin = end;
      const uint16_t* lo[3] = {w.lox, w.loy, w.loz};
      const uint16_t* hi[3] = {w.hix, w.hiy, w.hiz};
      const float org[3] = {w.ox, w.oy, w.oz};
      for (int a = 0; a < 3; a++) {
        const float step = quant_step(w.exps >> (8 * a));
        if (b.lo[a] <= b.hi[a])
          errors += !(dequant(plane_value(lo[a][s]), step, org[a]) <= b.lo[a] && dequant(plane_value(hi[a][s]), step, org[a]) >= b.hi[a]);
        nb.lo[a] = std::min(nb.lo[a], b.lo[a]);
        nb.hi[a] = std::max(nb.hi[a], b.hi[a]);
      }
    }
    need[x] += inner > 1 ? 1 : 0;
    box[x] = nb;
  }
  for (uint32_t r : reached) errors += r != 1;
  out[0] = uint32_t(wide.size());
  out[1] = need[0];
  out[2] = BvhStackNeed(nodes);
  return errors;
}

extern "C" uint32_t probe_wide_host(const float* bounds, uint32_t n, int max_leaf, uint32_t out[3]) {
  BvhBuildResult r;
  BuildBvh4Host(bounds, n, max_leaf, r);
  return Wide(r.nodes, bounds, r.order, out);
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
  return Wide(nodes, bounds.data(), order, out);
}
