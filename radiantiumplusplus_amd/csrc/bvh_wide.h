// The traversal's 8-wide nodes from a BvhNode4 tree, node by node (host and
// device): which children a node takes, their slots, the quantised planes and
// the places of the primitives.  bvh_gpu.hip runs it level by level.
#pragma once

#include <cmath>
#include <cstddef>
#include <cstdint>

#include "scene_dev.h"

namespace rad {

// A node to make: a BvhNode4 with its inner children opened while they fit, or
// one node of a chain.  A BvhNode4 whose leaves hold more than kWideNodePrims
// primitives becomes a chain of nodes: each takes leaves up to that many, and
// its one inner child is the node of all that is left, the inner children
// among it.  A chain node never has two inner children, so the stack of a
// traversal holds no more than the BvhNode4 tree asks for.
struct WideJob {
  uint32_t n4;
  uint32_t mask;   // children of n4 still to be placed, bits 0-3; kWideRest: not the first of its chain
  uint32_t skip;   // primitives of the first of them that the chain has placed already (a leaf of more than kWideNodePrims)
  uint32_t begin;  // with kWideRest: place of its first primitive, reserved by the chain's first node
};
constexpr uint32_t kWideAll = 15u, kWideRest = 16u, kWideNone = 0xffffffffu;

// The children of a node: BvhNode4 * 4 + child, kWideNone for none.  A chain
// node has its leaves or inner children at 0-3 and the rest of its chain at 4.
struct WideKids {
  uint32_t k[8];
};

RAD_HD float half_area(const float lo[3], const float hi[3]) {
  const float dx = hi[0] - lo[0], dy = hi[1] - lo[1], dz = hi[2] - lo[2];
  if (!(dx >= 0.f && dy >= 0.f && dz >= 0.f)) return 0.f;
  return dx * dy + dy * dz + dz * dx;
}

RAD_HD void slot_box(const BvhNode4* nodes, uint32_t kid, float lo[3], float hi[3]) {
  const BvhNode4& nd = nodes[kid >> 2];
  const uint32_t s = kid & 3u;
  lo[0] = nd.lox[s], lo[1] = nd.loy[s], lo[2] = nd.loz[s];
  hi[0] = nd.hix[s], hi[1] = nd.hiy[s], hi[2] = nd.hiz[s];
}

// The primitives of the leaves among the children `mask` of a BvhNode4.
RAD_HD uint32_t leaf_total(const BvhNode4& nd, uint32_t mask) {
  uint32_t prims = 0;
  for (uint32_t s = 0; s < 4; s++)
    if ((mask >> s & 1u) && nd.child[s] >= 0) prims += nd.count[s];
  return prims;
}
RAD_HD bool is_chain(const BvhNode4& nd, const WideJob& jb) {
  return (jb.mask & kWideRest) || leaf_total(nd, kWideAll) > kWideNodePrims;
}

// The children of a node that is no chain node: the BvhNode4's own four, then
// the inner one of largest area replaced by its children while at most eight
// result and their leaves hold at most kWideNodePrims primitives.
__host__ __device__ inline int wide_children(const BvhNode4* nodes, uint32_t root, uint32_t out[8]) {
  int n = 0;
  uint32_t prims = 0;
  for (uint32_t s = 0; s < 4; s++)
    if (nodes[root].child[s] >= 0) {
      prims += nodes[root].count[s];
      out[n++] = root * 4 + s;
    }
  for (;;) {
    int best = -1;
    float area = -1.f;
    uint32_t bestPrims = 0;
    for (int i = 0; i < n; i++) {
      const BvhNode4& nd = nodes[out[i] >> 2];
      if (nd.count[out[i] & 3u] > 0) continue;
      const BvhNode4& c = nodes[nd.child[out[i] & 3u]];
      int k = 0;
      uint32_t p = 0;
      for (int s = 0; s < 4; s++)
        if (c.child[s] >= 0) {
          k++;
          p += c.count[s];
        }
      if (n - 1 + k > 8 || prims + p > kWideNodePrims) continue;
      float lo[3], hi[3];
      slot_box(nodes, out[i], lo, hi);
      const float a = half_area(lo, hi);
      if (a > area) {
        area = a;
        best = i;
        bestPrims = p;
      }
    }
    if (best < 0) return n;
    const uint32_t c = uint32_t(nodes[out[best] >> 2].child[out[best] & 3u]);
    prims += bestPrims;
    bool first = true;
    for (uint32_t s = 0; s < 4; s++)
      if (nodes[c].child[s] >= 0) {
        out[first ? best : n++] = c * 4 + s;
        first = false;
      }
  }
}

// The children of a chain node and how many primitives it takes of each leaf
// (0: inner); rest: the job of what is left, child 4, if any.  A leaf of which a
// part is placed has its parts in nodes of their own, one after the other, so
// that its primitives stay consecutive.  Every node places primitives or the
// last inner children, so a chain ends.
__host__ __device__ inline void chain_children(const BvhNode4& nd, const WideJob& jb, uint32_t kid[8], uint32_t cnt[8],
                                               WideJob& rest) {
  for (int i = 0; i < 8; i++) kid[i] = kWideNone, cnt[i] = 0;
  uint32_t left = 0, acc = 0;  // children still to be placed, primitives taken
  for (uint32_t s = 0; s < 4; s++) left |= nd.child[s] >= 0 ? jb.mask & 1u << s : 0u;
  rest = WideJob{jb.n4, 0, 0, 0};
  const bool end = jb.skip == 0 && leaf_total(nd, left) <= kWideNodePrims;  // the last leaves and the inner children
  bool part = false;                                                        // a part of a large leaf, by itself
  for (uint32_t s = 0; s < 4; s++) {
    if (!(left >> s & 1u) || (!end && nd.count[s] == 0) || part) continue;
    const uint32_t c = nd.count[s] - (acc == 0 ? jb.skip : 0u);  // the first leaf is the one begun
    if (acc == 0 && (jb.skip || c > kWideNodePrims)) part = true;
    if (!part && acc + c > kWideNodePrims) continue;
    kid[s] = jb.n4 * 4 + s;
    cnt[s] = c < kWideNodePrims ? c : kWideNodePrims;
    acc += cnt[s];
    if (c > kWideNodePrims)
      rest.skip = jb.skip + kWideNodePrims;
    else
      left &= ~(1u << s);
  }
  if (left) {
    kid[4] = jb.n4 * 4;
    rest.mask = left | kWideRest;
  }
}

// slot[i]: the slot of child i (of those in `valid`), chosen greedily so that
// bit a of a slot says on which side of the node's centre the child's centre
// lies along axis a.
RAD_HD void wide_order(const float l[3][8], const float h[3][8], uint32_t valid, const float lo[3], const float hi[3],
                       uint32_t slot[8]) {
  float d[3][8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    for (int a = 0; a < 3; a++) d[a][i] = (l[a][i] + h[a][i]) - (lo[a] + hi[a]);
    slot[i] = 0;
  }
  // each child's best free slot; after a choice only children that wanted the
  // same slot look again
  float c[8];
  uint32_t want[8], used = 0, todo = valid, again = valid;
  while (todo) {
    uint32_t bi = 8;
    float best = -kInf;
#pragma unroll
    for (uint32_t i = 0; i < 8; i++) {
      if (again >> i & 1u) {
        want[i] = 8;
#pragma unroll
        for (uint32_t s = 0; s < 8; s++) {
          const float v = (s & 1 ? d[0][i] : -d[0][i]) + (s & 2 ? d[1][i] : -d[1][i]) + (s & 4 ? d[2][i] : -d[2][i]);
          if (!(used >> s & 1u) && (want[i] == 8 || v > c[i])) c[i] = v, want[i] = s;
        }
      }
      if ((todo >> i & 1u) && (bi == 8 || c[i] > best)) best = c[i], bi = i;
    }
    uint32_t bs = 0;
#pragma unroll
    for (uint32_t i = 0; i < 8; i++) {
      bs = i == bi ? want[i] : bs;
      slot[i] = i == bi ? want[i] : slot[i];
    }
    todo &= ~(1u << bi);
    used |= 1u << bs;
    again = 0;
#pragma unroll
    for (uint32_t i = 0; i < 8; i++) again |= (todo >> i & 1u) && want[i] == bs ? 1u << i : 0u;
  }
}

// Step 2^e of one axis, e the smallest with kWidePlaneMax * 2^e >= the node's
// extent (raised further if rounding keeps a bound out of reach), and the
// children's planes qlo, qhi in it, rounded outward and verified with the
// traversal's own dequantisation.
RAD_HD bool quantize_axis(const float clo[8], const float chi[8], uint32_t valid, float o, float ext, uint32_t& biased,
                          uint32_t qlo[8], uint32_t qhi[8]) {
  constexpr float top = float(kWidePlaneMax);
  int e = -126;
  if (ext > 0.f) {
    frexpf(ext / top, &e);  // ext / top = m 2^e, m in [0.5, 1)
    e = e > -126 ? e : -126;
  }
  for (; e <= 127; e++) {
    biased = uint32_t(e + 127);
    const float step = quant_step(biased), inv = biased < 254 ? quant_step(254 - biased) : 0x1p-127f;  // 1 / step
    bool ok = true;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      if (!(valid >> i & 1u)) continue;
      const float y = fminf(fmaxf((chi[i] - o) * inv, 0.f), top);
      uint32_t a = uint32_t(fminf(fmaxf((clo[i] - o) * inv, 0.f), top)), c = uint32_t(y);
      if (float(c) < y) c++;
      while (a > 0 && dequant(a, step, o) > clo[i]) a--;
      while (c < kWidePlaneMax && dequant(c, step, o) < chi[i]) c++;
      if (!(dequant(a, step, o) <= clo[i] && dequant(c, step, o) >= chi[i])) ok = false;
      qlo[i] = a;
      qhi[i] = c;
    }
    if (ok) return true;
  }
  return false;
}

// The planes of eight slots from those of the children, to the 16-byte chunk
// `out`.
RAD_HD void place_planes(const uint32_t q[8], const uint32_t slot[8], uint32_t valid, uint32_t empty, char* out) {
  uint32_t w[4] = {0, 0, 0, 0}, used = 0;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    if (!(valid >> i & 1u)) continue;
    const uint32_t b = uint32_t(plane_bits(q[i])) << (16 * (slot[i] & 1u));
    used |= 1u << slot[i];
#pragma unroll
    for (uint32_t v = 0; v < 4; v++) w[v] |= slot[i] >> 1 == v ? b : 0u;
  }
#pragma unroll
  for (uint32_t s = 0; s < 8; s++) w[s >> 1] |= used >> s & 1u ? 0u : empty << (16 * (s & 1u));
  __builtin_memcpy(__builtin_assume_aligned(out, 16), w, 16);
}

// First pass over a job: its children go to `kids`; returns how many of them
// are inner (low word) and how many primitives it reserves (high word).
__host__ __device__ inline unsigned long long wide_count(const BvhNode4* nodes, const WideJob& jb, WideKids& kids) {
  uint32_t inner = 0, prims = 0;
  if (is_chain(nodes[jb.n4], jb)) {
    uint32_t cnt[8];
    WideJob rest;
    chain_children(nodes[jb.n4], jb, kids.k, cnt, rest);
    for (int i = 0; i < 8; i++) inner += kids.k[i] != kWideNone && cnt[i] == 0 ? 1u : 0u;
    if (!(jb.mask & kWideRest)) prims = leaf_total(nodes[jb.n4], kWideAll);
  } else {
    uint32_t w[8];
    const int n = wide_children(nodes, jb.n4, w);
    for (int i = 0; i < 8; i++) {
      kids.k[i] = i < n ? w[i] : kWideNone;
      if (i >= n) continue;
      const uint32_t c = nodes[w[i] >> 2].count[w[i] & 3u];
      inner += c == 0 ? 1u : 0u;
      prims += c;
    }
  }
  return (static_cast<unsigned long long>(prims) << 32) | inner;
}

// Second pass: the node, the jobs of its inner children (next, in slot order;
// their nodes are child0, child0 + 1, ...), the new places of its primitives
// from prim0 on (perm: where each is now), and those places in the leaves of
// the BvhNode4 tree.  Returns false if a child box cannot be bounded.
//
// Bound by the latency of one thread's steps: the levels of a tree follow each
// other and most are small.  Every array is indexed by constants, so that none
// is in scratch memory or read through a loop over lanes, and the axes share
// their code, which a launch reads anew (60 KB with three copies, now 31; 2.6 M
// primitives, 12 levels: 980 us with arrays indexed by slot, now 501).
RAD_HD bool wide_emit(BvhNode4* nodes, WideJob jb, const WideKids& kids, uint32_t child0, uint32_t prim0, BvhNode8* out,
                      WideJob* next, uint32_t* perm) {
  const WideKids kd = kids;
  const bool chain = is_chain(nodes[jb.n4], jb);
  uint32_t cnt[8], valid = 0;  // cnt: primitives of a leaf, 0: inner
  WideJob rest{};
#pragma unroll
  for (int i = 0; i < 8; i++) {
    valid |= kd.k[i] != kWideNone ? 1u << i : 0u;
    cnt[i] = kd.k[i] != kWideNone ? nodes[kd.k[i] >> 2].count[kd.k[i] & 3u] : 0u;
  }
  if (chain) {
    uint32_t k[8];
    chain_children(nodes[jb.n4], jb, k, cnt, rest);
  }
  float l[3][8], h[3][8], lo[3] = {kInf, kInf, kInf}, hi[3] = {-kInf, -kInf, -kInf};
#pragma unroll
  for (int i = 0; i < 8; i++) {
    float bl[3] = {kInf, kInf, kInf}, bh[3] = {-kInf, -kInf, -kInf};
    if (chain && i == 4) {
      for (uint32_t s = 0; s < 4; s++)
        if (rest.mask >> s & 1u) {
          float tl[3], th[3];
          slot_box(nodes, jb.n4 * 4 + s, tl, th);
          for (int a = 0; a < 3; a++) bl[a] = fminf(bl[a], tl[a]), bh[a] = fmaxf(bh[a], th[a]);
        }
    } else if (valid >> i & 1u) {
      slot_box(nodes, kd.k[i], bl, bh);
    }
    for (int a = 0; a < 3; a++) {
      l[a][i] = bl[a], h[a][i] = bh[a];
      lo[a] = fminf(lo[a], bl[a]), hi[a] = fmaxf(hi[a], bh[a]);
    }
  }
  uint32_t slot[8];
  wide_order(l, h, valid, lo, hi, slot);
  uint32_t imask = 0, total = 0, ends[2] = {0, 0};
#pragma unroll
  for (int i = 0; i < 8; i++) {
    if (!(valid >> i & 1u)) continue;
    imask |= cnt[i] == 0 ? 1u << slot[i] : 0u;
    total += cnt[i];
#pragma unroll
    for (uint32_t s = 0; s < 8; s++) ends[s >> 2] += slot[i] <= s ? cnt[i] << (8 * (s & 3u)) : 0u;
  }
  rest.begin = prim0 + total;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    if (!(valid >> i & 1u)) continue;
    if (cnt[i] == 0) {
      WideJob j{0, kWideAll, 0, 0};
      if (chain && i == 4)
        j = rest;
      else
        j.n4 = uint32_t(nodes[kd.k[i] >> 2].child[kd.k[i] & 3u]);
      next[__builtin_popcount(imask & ((1u << slot[i]) - 1u))] = j;
      continue;
    }
    uint32_t begin = prim0;
#pragma unroll
    for (int k = 0; k < 8; k++) begin += (valid >> k & 1u) && slot[k] < slot[i] ? cnt[k] : 0u;
    BvhNode4& leaf = nodes[kd.k[i] >> 2];
    const uint32_t s = kd.k[i] & 3u, skip = chain ? jb.skip : 0u;  // a leaf of which a part was placed is the only one here
    const uint32_t from = uint32_t(leaf.child[s]) + skip;
    for (uint32_t q = 0; q < cnt[i]; q++) perm[begin + q] = from + q;
    if (!chain || skip + cnt[i] == leaf.count[s]) leaf.child[s] = int32_t(begin - skip);
  }
  // one axis after the other through the same code
  static_assert(offsetof(BvhNode8, lox) == 0 && offsetof(BvhNode8, hix) == 16 && offsetof(BvhNode8, loz) == 48 &&
                    offsetof(BvhNode8, loy) == 64 && offsetof(BvhNode8, hiy) == 96 && offsetof(BvhNode8, hiz) == 112,
                "plane chunks");
  char* const chunk = reinterpret_cast<char*>(out);
  uint32_t exps = imask << 24;
  out->ox = lo[0];
  out->oy = lo[1];
  out->oz = lo[2];
  bool ok = true;
#pragma nounroll
  for (int a = 0; a < 3; a++) {
    uint32_t biased = 127, q[2][8] = {};
    ok = quantize_axis(l[0], h[0], valid, lo[0], hi[0] - lo[0], biased, q[0], q[1]) && ok;
    exps |= (biased & 0xffu) << (8 * a);
    // an empty slot: an inverted box
    place_planes(q[0], slot, valid, plane_bits(kWidePlaneMax), chunk + (a == 0 ? 0 : a == 1 ? 64 : 48));
    place_planes(q[1], slot, valid, 0, chunk + (a == 0 ? 16 : a == 1 ? 96 : 112));
#pragma unroll
    for (int i = 0; i < 8; i++) {
      l[0][i] = l[1][i], l[1][i] = l[2][i];
      h[0][i] = h[1][i], h[1][i] = h[2][i];
    }
    lo[0] = lo[1], lo[1] = lo[2];
    hi[0] = hi[1], hi[1] = hi[2];
  }
  out->exps = exps;
  out->child_base = child0;
  out->prim_base = prim0;
  out->ends[0] = ends[0];
  out->ends[1] = ends[1];
  return ok;
}

}  // namespace rad
