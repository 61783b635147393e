// Device BVH build (replaces the Embree build, embree.cpp:18-43).
//
// 1. Centroids are ordered along a 63-bit Morton curve (hipCUB radix sort):
//    the starting order, so neighbouring lanes hold nearby primitives.
// 2. Top-down, one level of nodes at a time over the whole GPU.  A node
//    with more than kSmall primitives is split by binned SAH: 16 centroid
//    bins on each axis, summed in LDS per chunk of primitives, the best axis and bin boundary chosen
//    by the surface-area heuristic, and the node's range partitioned stably
//    in place through a prefix sum of the go-left flags.  Nodes of at most
//    kSmall primitives are built to the leaves by one wave each, with an
//    exact SAH sweep over the centroid order of every axis.  Ranges of at
//    most max_leaf primitives become leaves.
// 3. The binary tree is collapsed into 4-wide nodes (repeatedly opening the
//    inner child of largest area), again level by level.
// 4. The traversal's 8-wide quantised nodes are made from the 4-wide tree of
//    either builder, level by level, with the primitives put in the order of
//    its leaves.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <chrono>
#include <stdexcept>

#include "bvh_gpu.h"
#include "bvh_wide.h"

namespace rad {
namespace {

constexpr uint32_t kNone = 0xffffffffu;
constexpr int kBins = 16;
constexpr uint32_t kSmall = 64;

struct N2 {
  float lo[3];
  uint32_t left;   // inner: first of two consecutive children; leaf: first sorted primitive
  float hi[3];
  uint32_t count;  // 0: inner
};

__device__ __forceinline__ void atomic_min_f(float* a, float v) {
  if (v >= 0.f)
    atomicMin(reinterpret_cast<int*>(a), __float_as_int(v));
  else
    atomicMax(reinterpret_cast<unsigned int*>(a), __float_as_uint(v));
}
__device__ __forceinline__ void atomic_max_f(float* a, float v) {
  if (v >= 0.f)
    atomicMax(reinterpret_cast<int*>(a), __float_as_int(v));
  else
    atomicMin(reinterpret_cast<unsigned int*>(a), __float_as_uint(v));
}

// Minimum / maximum over the wave, in every lane (all 64 lanes active): data
// parallel moves within and across rows instead of LDS permutes.
template <bool MAX>
__device__ __forceinline__ float wave_extreme(float v) {
  const auto step = [](float x, float y) { return MAX ? fmaxf(x, y) : fminf(x, y); };
#define RAD_DPP(ctrl, rows) \
  v = step(v, __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), ctrl, rows, 0xf, false)))
  RAD_DPP(0x111, 0xf);  // row_shr:1
  RAD_DPP(0x112, 0xf);
  RAD_DPP(0x114, 0xf);
  RAD_DPP(0x118, 0xf);
  RAD_DPP(0x142, 0xa);  // row_bcast:15
  RAD_DPP(0x143, 0xc);  // row_bcast:31
#undef RAD_DPP
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
__device__ __forceinline__ float wave_min(float v) { return wave_extreme<false>(v); }
__device__ __forceinline__ float wave_max(float v) { return wave_extreme<true>(v); }

// Unsigned integers in the order of the floats, for LDS minima and maxima.
__device__ __forceinline__ uint32_t ordered_bits(float v) {
  const uint32_t u = __float_as_uint(v);
  return u ^ (uint32_t(int32_t(u) >> 31) | 0x80000000u);
}
__device__ __forceinline__ float from_ordered(uint32_t u) {
  return __uint_as_float(u ^ (uint32_t(int32_t(~u) >> 31) | 0x80000000u));
}

// ---------------------------------------------------------------- ordering
// A fixed grid, so that the six atomics per wave stay few: with one wave per
// 64 primitives they took 2.8 ms on 2.6 M primitives (about 11 ns each).
__global__ void k_centroid_bounds(const float* b, uint32_t n, float* cb) {
  float lo[3] = {kInf, kInf, kInf}, hi[3] = {-kInf, -kInf, -kInf};
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    for (int a = 0; a < 3; a++) {
      const float c = 0.5f * (b[6 * size_t(i) + a] + b[6 * size_t(i) + 3 + a]);
      lo[a] = fminf(lo[a], c);
      hi[a] = fmaxf(hi[a], c);
    }
  for (int a = 0; a < 3; a++) lo[a] = wave_min(lo[a]), hi[a] = wave_max(hi[a]);
  if (__lane_id() == 0)
    for (int a = 0; a < 3; a++) {
      atomic_min_f(&cb[a], lo[a]);
      atomic_max_f(&cb[3 + a], hi[a]);
    }
}

// Primitive records and boxes: triangles from the scene's per-triangle
// records, other shapes (one primitive each) as the host made them.
__global__ void k_primitives(const PrimSegment* segs, uint32_t nSegs, const float4* tris, const float4* otherRec,
                             const float* otherBox, uint32_t n, float4* rec, float* box) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint32_t l = 0, r = nSegs;  // the last segment that begins at or before i
  while (r - l > 1) {
    const uint32_t m = (l + r) / 2;
    if (segs[m].begin <= i)
      l = m;
    else
      r = m;
  }
  const PrimSegment sg = segs[l];
  float4* o = rec + 3 * size_t(i);
  float* q = box + 6 * size_t(i);
  if (sg.other != kNone) {
    for (int k = 0; k < 3; k++) o[k] = otherRec[3 * size_t(sg.other) + k];
    for (int k = 0; k < 6; k++) q[k] = otherBox[6 * size_t(sg.other) + k];
    return;
  }
  const uint32_t t = i - sg.begin;
  const float4* s = tris + 6 * (size_t(sg.tri_offset) + t);
  const float4 a = s[0], b = s[1], c = s[2];
  const float v[3][3] = {{a.x, a.y, a.z}, {a.w, b.x, b.y}, {b.z, b.w, c.x}};
  o[0] = make_float4(v[0][0], v[0][1], v[0][2], __uint_as_float(sg.geom));
  o[1] = make_float4(v[1][0], v[1][1], v[1][2], __uint_as_float(t));
  o[2] = make_float4(v[2][0], v[2][1], v[2][2], __uint_as_float(PRIM_TRI));
  for (int k = 0; k < 3; k++) {
    q[k] = fminf(fminf(v[0][k], v[1][k]), v[2][k]);
    q[3 + k] = fmaxf(fmaxf(v[0][k], v[1][k]), v[2][k]);
  }
}

__device__ __forceinline__ uint64_t spread21(uint32_t v) {
  uint64_t x = v & 0x1fffffu;
  x = (x | x << 32) & 0x1f00000000ffffull;
  x = (x | x << 16) & 0x1f0000ff0000ffull;
  x = (x | x << 8) & 0x100f00f00f00f00full;
  x = (x | x << 4) & 0x10c30c30c30c30c3ull;
  x = (x | x << 2) & 0x1249249249249249ull;
  return x;
}

__global__ void k_morton(const float* b, uint32_t n, const float* cb, uint64_t* keys, uint32_t* ids) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint32_t q[3];
  for (int a = 0; a < 3; a++) {
    float c = 0.5f * (b[6 * size_t(i) + a] + b[6 * size_t(i) + 3 + a]);
    float e = cb[3 + a] - cb[a];
    float t = e > 0.f ? (c - cb[a]) / e : 0.5f;
    q[a] = uint32_t(fminf(fmaxf(t, 0.f), 1.f) * 2097151.f);
  }
  keys[i] = spread21(q[0]) | spread21(q[1]) << 1 | spread21(q[2]) << 2;
  ids[i] = i;
}

// sorted SoA bounds: lo.xyz + pad, hi.xyz + pad
__global__ void k_gather_bounds(const float* b, const uint32_t* ids, uint32_t n, float4* blo, float4* bhi) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float* s = b + 6 * size_t(ids[i]);
  blo[i] = make_float4(s[0], s[1], s[2], 0.f);
  bhi[i] = make_float4(s[3], s[4], s[5], 0.f);
}

// ---------------------------------------------------------------- top-down build
// Large nodes (more than kSmall primitives) are split one level at a time
// over the whole GPU: their primitives add their boxes to 16 centroid bins
// on each axis, the surface-area heuristic picks the axis and bin boundary,
// and a flag scan partitions the node's range in place (stable, ping-pong
// buffers).  Nodes of at most kSmall primitives are finished by one wave
// each with an exact SAH sweep over every centroid on every axis.
struct Task {
  uint32_t node, begin, end, nl;  // nl: primitives going left (set by the split)
  float clo[3];
  uint32_t axis;                  // split axis; 3: median split of the current order
  float chi[3];
  uint32_t kbin;                  // first bin of the right child
  uint32_t child_task[2];         // next-level task of each child, kNone if it is a leaf or small
  uint32_t pad[2];
};

struct SmallTask {
  uint32_t node, begin, end;
  uint32_t nodes;  // 2 * (end - begin - 1) nodes reserved for the subtree
};

struct Bin {
  float lo[3];
  uint32_t count;
  float hi[3];
  uint32_t pad;
};

struct BuildCtr {
  uint32_t nodes;   // binary nodes allocated
  uint32_t tasks;   // large tasks of the next level
  uint32_t smalls;  // small tasks (all levels)
  uint32_t error;   // set when a capacity would be exceeded (nothing is written then)
};

struct Caps {
  uint32_t nodes, tasks, smalls;
};

__device__ __forceinline__ int bin_of(float c, float lo, float hi) {
  const float e = hi - lo;
  if (!(e > 0.f)) return 0;
  const int k = int((c - lo) * (float(kBins) / e));
  return min(max(k, 0), kBins - 1);
}

__device__ __forceinline__ float4 centroid(float4 lo, float4 hi) {
  return make_float4(0.5f * (lo.x + hi.x), 0.5f * (lo.y + hi.y), 0.5f * (lo.z + hi.z), 0.f);
}
__device__ __forceinline__ float comp(float4 v, int a) { return a == 0 ? v.x : a == 1 ? v.y : v.z; }

__global__ void k_bins_clear(Bin* bins, uint32_t m) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  Bin e;
  for (int a = 0; a < 3; a++) {
    e.lo[a] = kInf;
    e.hi[a] = -kInf;
  }
  e.count = 0;
  e.pad = 0;
  bins[i] = e;
}

// The level passes work on chunks of kLevelChunk consecutive primitives per
// block.  A large task's primitives are consecutive and more than kSmall, so a
// chunk meets at most kLevelSlots of them: sums go to LDS by (task of the
// chunk, bin) and then to memory once per chunk, instead of once per wave and
// bin (2.6 M primitives, 21 levels: binning 12.7 ms, child centroid bounds 9.4
// ms, most of it waiting on atomics to a few addresses).
constexpr int kLevelThreads = 256, kLevelItems = 4;
constexpr uint32_t kLevelChunk = kLevelThreads * kLevelItems;
constexpr uint32_t kLevelSlots = kLevelChunk / (kSmall + 1) + 2;

// t[e]: task of item blockIdx.x * kLevelChunk + e * kLevelThreads + threadIdx.x
// (kNone: none), slot[e]: its number among the chunk's tasks, sTask: the
// chunk's tasks.  Returns how many there are.
__device__ __forceinline__ uint32_t chunk_slots(uint32_t n, const uint32_t* owner, uint32_t t[kLevelItems],
                                                uint32_t slot[kLevelItems], uint32_t* sTask, BuildCtr* ctr) {
  __shared__ uint32_t sHeads[kLevelItems * kLevelThreads / 64];
  const uint32_t base = blockIdx.x * kLevelChunk, wave = threadIdx.x >> 6, lane = __lane_id();
  uint64_t heads[kLevelItems];
#pragma unroll
  for (int e = 0; e < kLevelItems; e++) {
    const uint32_t i = base + e * kLevelThreads + threadIdx.x;
    t[e] = i < n ? owner[i] : kNone;
    const bool head = t[e] != kNone && (i == base || owner[i - 1] != t[e]);
    heads[e] = __ballot(head);
    if (lane == 0) sHeads[e * (kLevelThreads / 64) + wave] = uint32_t(__popcll(heads[e]));
  }
  __syncthreads();
  uint32_t total = 0;
#pragma unroll
  for (int e = 0; e < kLevelItems; e++)
    for (uint32_t v = 0; v < kLevelThreads / 64; v++) {
      if (v == wave) slot[e] = total + uint32_t(__popcll(heads[e] & (~0ull >> (63 - lane)))) - 1u;
      total += sHeads[e * (kLevelThreads / 64) + v];
    }
#pragma unroll
  for (int e = 0; e < kLevelItems; e++) {
    if (t[e] == kNone) continue;
    if (slot[e] >= kLevelSlots) {  // not a partition into ranges of more than kSmall: report, leave it out
      atomicOr(&ctr->error, 16u);
      t[e] = kNone;
    } else if (heads[e] >> lane & 1ull) {
      sTask[slot[e]] = t[e];
    }
  }
  __syncthreads();
  return min(total, kLevelSlots);
}

// LDS sums of one key: box (6 ordered words) and, with COUNT, a count.
template <bool COUNT>
__device__ __forceinline__ void lds_add(uint32_t* s, const float lo[3], const float hi[3], uint32_t count) {
  for (int a = 0; a < 3; a++) {
    atomicMin(&s[a], ordered_bits(lo[a]));
    atomicMax(&s[3 + a], ordered_bits(hi[a]));
  }
  if (COUNT) atomicAdd(&s[6], count);
}
// Adds this lane's box to sums[key] (kNone: nothing).  The two commonest cases,
// a wave with one or two keys, are combined in registers first; the lanes left
// over then meet in few places and add theirs one by one.
template <bool COUNT>
__device__ __forceinline__ void wave_add(uint32_t* sums, uint32_t key, const float lo[3], const float hi[3]) {
  constexpr uint32_t W = COUNT ? 7 : 6;
  uint64_t pending = __ballot(key != kNone);
  for (int pass = 0; pass < 2 && pending; pass++) {
    const int leader = __ffsll((unsigned long long)pending) - 1;
    const uint32_t target = __builtin_amdgcn_readlane(key, leader);
    const bool mine = key == target;
    const uint64_t group = __ballot(mine);
    if (__popcll(group) < 12) break;
    pending &= ~group;
    float l[3], h[3];
    for (int a = 0; a < 3; a++) {
      l[a] = wave_min(mine ? lo[a] : kInf);
      h[a] = wave_max(mine ? hi[a] : -kInf);
    }
    if (__lane_id() == uint32_t(leader)) lds_add<COUNT>(sums + W * target, l, h, uint32_t(__popcll(group)));
  }
  if (pending >> __lane_id() & 1ull) lds_add<COUNT>(sums + W * key, lo, hi, 1u);
}

// Every primitive of a large node adds its box to one bin per axis.
__global__ void __launch_bounds__(kLevelThreads) k_bins_accum(uint32_t n, const uint32_t* owner, const Task* tasks,
                                                              const float4* blo, const float4* bhi, Bin* bins,
                                                              BuildCtr* ctr) {
  __shared__ uint32_t sSum[kLevelSlots * 3 * kBins * 7], sTask[kLevelSlots];
  uint32_t t[kLevelItems], slot[kLevelItems];
  const uint32_t slots = chunk_slots(n, owner, t, slot, sTask, ctr);
  if (slots == 0) return;
  for (uint32_t j = threadIdx.x; j < slots * 3 * kBins * 7; j += kLevelThreads)
    sSum[j] = j % 7 < 3 ? ordered_bits(kInf) : j % 7 < 6 ? ordered_bits(-kInf) : 0u;
  __syncthreads();
  for (int e = 0; e < kLevelItems; e++) {
    float lo[3] = {kInf, kInf, kInf}, hi[3] = {-kInf, -kInf, -kInf};
    int k[3] = {0, 0, 0};
    if (t[e] != kNone) {
      const uint32_t i = blockIdx.x * kLevelChunk + e * kLevelThreads + threadIdx.x;
      const Task& tk = tasks[t[e]];
      const float4 l = blo[i], h = bhi[i], c = centroid(l, h);
      lo[0] = l.x, lo[1] = l.y, lo[2] = l.z;
      hi[0] = h.x, hi[1] = h.y, hi[2] = h.z;
      k[0] = bin_of(c.x, tk.clo[0], tk.chi[0]);
      k[1] = bin_of(c.y, tk.clo[1], tk.chi[1]);
      k[2] = bin_of(c.z, tk.clo[2], tk.chi[2]);
    }
    for (int a = 0; a < 3; a++) wave_add<true>(sSum, t[e] == kNone ? kNone : (slot[e] * 3 + a) * kBins + k[a], lo, hi);
  }
  __syncthreads();
  for (uint32_t j = threadIdx.x; j < slots * 3 * kBins; j += kLevelThreads) {
    const uint32_t* s = sSum + 7 * j;
    if (s[6] == 0) continue;
    Bin* e = &bins[size_t(sTask[j / (3 * kBins)]) * 3 * kBins + j % (3 * kBins)];
    for (int a = 0; a < 3; a++) {
      atomic_min_f(&e->lo[a], from_ordered(s[a]));
      atomic_max_f(&e->hi[a], from_ordered(s[3 + a]));
    }
    atomicAdd(&e->count, s[6]);
  }
}

// One wave per large task: best binned SAH split over the three axes, children
// allocated; a child of one primitive becomes a leaf, one of at most kSmall a
// small task (its subtree's nodes reserved with it), a larger one a task of the
// next level.  Lane 16 a + k holds bin k of axis a: prefixes and suffixes over
// an axis are scans within a row of 16 lanes (one thread per task walked the
// 48 bins from memory in 34 us a level, whatever the number of tasks).
template <int CTRL, bool MAX>
__device__ __forceinline__ float row_step(float v) {
  const float o = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), CTRL, 0xf, 0xf, false));
  return MAX ? fmaxf(v, o) : fminf(v, o);
}
template <bool SUFFIX, bool MAX>
__device__ __forceinline__ float row_scan(float v) {  // row_shr for prefixes, row_shl for suffixes
  constexpr int base = SUFFIX ? 0x100 : 0x110;
  v = row_step<base + 1, MAX>(v);
  v = row_step<base + 2, MAX>(v);
  v = row_step<base + 4, MAX>(v);
  return row_step<base + 8, MAX>(v);
}
template <bool SUFFIX>
__device__ __forceinline__ uint32_t row_sum(uint32_t c) {
  constexpr int base = SUFFIX ? 0x100 : 0x110;
  int v = int(c);
  v += __builtin_amdgcn_update_dpp(0, v, base + 1, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, base + 2, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, base + 4, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, base + 8, 0xf, 0xf, false);
  return uint32_t(v);
}
__device__ __forceinline__ float prev_lane(float v, float first) {  // the value of the row's lane before, `first` at its start
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(first), __float_as_int(v), 0x111, 0xf, 0xf, false));
}
__device__ __forceinline__ float lane_f(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// The tasks of a block take their nodes and child tasks with one atomic each.
constexpr int kSplitWaves = 16;
__global__ void __launch_bounds__(64 * kSplitWaves) k_split(Task* tasks, uint32_t nTasks, const Bin* bins, N2* n2, Task* next,
                                                            SmallTask* smalls, BuildCtr* ctr, Caps caps) {
  __shared__ uint32_t sNeed[3][kSplitWaves], sBase[3];  // nodes, large and small child tasks
  const int wave = int(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
  const uint32_t t = blockIdx.x * kSplitWaves + uint32_t(wave);
  const bool valid = t < nTasks;
  const uint32_t lane = __lane_id();
  Task tk = tasks[valid ? t : nTasks - 1];
  const uint32_t cnt = tk.end - tk.begin;
  float bl[3] = {kInf, kInf, kInf}, bh[3] = {-kInf, -kInf, -kInf};
  uint32_t bc = 0;
  if (lane < 3 * kBins) {
    const Bin b = bins[size_t(valid ? t : nTasks - 1) * 3 * kBins + lane];
    for (int a = 0; a < 3; a++) bl[a] = b.lo[a], bh[a] = b.hi[a];
    bc = b.count;
  }
  float pl[3], ph[3], sl[3], sh[3];  // boxes of the bins before this one, of this one and those after it
  float lo[3], hi[3];
  for (int a = 0; a < 3; a++) {
    const float il = row_scan<false, false>(bl[a]), ih = row_scan<false, true>(bh[a]);
    lo[a] = lane_f(il, kBins - 1);
    hi[a] = lane_f(ih, kBins - 1);
    pl[a] = prev_lane(il, kInf);
    ph[a] = prev_lane(ih, -kInf);
    sl[a] = row_scan<true, false>(bl[a]);
    sh[a] = row_scan<true, true>(bh[a]);
  }
  const uint32_t pc = row_sum<false>(bc) - bc, sc = row_sum<true>(bc);
  float cost = kInf;
  if (lane < 3 * kBins && pc > 0 && sc > 0) cost = half_area(pl, ph) * float(pc) + half_area(sl, sh) * float(sc);
  const float best = wave_min(cost);
  const uint64_t at = __ballot(cost == best && best < kInf);
  const bool found = at != 0;
  const int win = found ? __ffsll((unsigned long long)at) - 1 : 0;
  const uint32_t axis = found ? uint32_t(win) / kBins : 3u, kbin = found ? uint32_t(win) % kBins : 0u;
  const uint32_t nl = found ? __builtin_amdgcn_readlane(pc, win) : cnt / 2;
  float clo[2][3], chi[2][3];  // children boxes
  for (int a = 0; a < 3; a++) {
    clo[0][a] = found ? lane_f(pl[a], win) : lo[a];
    chi[0][a] = found ? lane_f(ph[a], win) : hi[a];
    clo[1][a] = found ? lane_f(sl[a], win) : lo[a];
    chi[1][a] = found ? lane_f(sh[a], win) : hi[a];
  }
  const uint32_t cb[2] = {tk.begin, tk.begin + nl}, ce[2] = {tk.begin + nl, tk.end};
  uint32_t reserve[2], nLarge = 0, nSmall = 0;
  for (int s = 0; s < 2; s++) {
    const uint32_t m = ce[s] - cb[s];
    reserve[s] = m > 1 && m <= kSmall ? 2 * (m - 1) : 0;
    nSmall += reserve[s] ? 1u : 0u;
    nLarge += m > kSmall ? 1u : 0u;
  }
  if (lane == 0) {
    sNeed[0][wave] = valid ? 2u + reserve[0] + reserve[1] : 0u;
    sNeed[1][wave] = valid ? nLarge : 0u;
    sNeed[2][wave] = valid ? nSmall : 0u;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    uint32_t sum = 0;
    for (int v = 0; v < kSplitWaves; v++) {
      const uint32_t c = sNeed[threadIdx.x][v];
      sNeed[threadIdx.x][v] = sum;
      sum += c;
    }
    uint32_t* at = threadIdx.x == 0 ? &ctr->nodes : threadIdx.x == 1 ? &ctr->tasks : &ctr->smalls;
    sBase[threadIdx.x] = sum ? atomicAdd(at, sum) : 0u;
  }
  __syncthreads();
  if (lane != 0 || !valid) return;
  const uint32_t child = sBase[0] + sNeed[0][wave];
  uint32_t largeAt = sBase[1] + sNeed[1][wave], smallAt = sBase[2] + sNeed[2][wave];
  if (child + 2 + reserve[0] + reserve[1] > caps.nodes) {
    atomicOr(&ctr->error, 1u);
    tk.axis = 3;
    tk.nl = cnt / 2;
    tk.child_task[0] = tk.child_task[1] = kNone;
    tasks[t] = tk;
    return;
  }
  N2 me;
  for (int a = 0; a < 3; a++) me.lo[a] = lo[a], me.hi[a] = hi[a];
  me.left = child;
  me.count = 0;
  n2[tk.node] = me;
  for (int s = 0; s < 2; s++) {
    const uint32_t m = ce[s] - cb[s];
    tk.child_task[s] = kNone;
    if (m == 1) {
      N2 leaf;
      for (int a = 0; a < 3; a++) leaf.lo[a] = clo[s][a], leaf.hi[a] = chi[s][a];
      leaf.left = cb[s];
      leaf.count = m;
      n2[child + s] = leaf;
    } else if (m <= kSmall) {  // the wave builder also decides leaves of at most max_leaf
      const uint32_t j = smallAt++;
      if (j >= caps.smalls) {
        atomicOr(&ctr->error, 2u);
        continue;
      }
      smalls[j] = SmallTask{child + s, cb[s], ce[s], child + 2 + (s ? reserve[0] : 0u)};
    } else {
      const uint32_t j = largeAt++;
      if (j >= caps.tasks) {
        atomicOr(&ctr->error, 4u);
        continue;
      }
      Task c;
      c.node = child + s;
      c.begin = cb[s];
      c.end = ce[s];
      c.nl = 0;
      c.axis = 3;
      c.kbin = 0;
      for (int a = 0; a < 3; a++) c.clo[a] = kInf, c.chi[a] = -kInf;
      c.child_task[0] = c.child_task[1] = kNone;
      c.pad[0] = c.pad[1] = 0;
      next[j] = c;
      tk.child_task[s] = j;
    }
  }
  tk.axis = axis;
  tk.kbin = kbin;
  tk.nl = nl;
  tasks[t] = tk;
}

__device__ __forceinline__ bool goes_left(const Task& tk, uint32_t i, float4 lo, float4 hi) {
  if (tk.axis >= 3) return i - tk.begin < tk.nl;
  const float4 c = centroid(lo, hi);
  return bin_of(comp(c, int(tk.axis)), tk.clo[tk.axis], tk.chi[tk.axis]) < int(tk.kbin);
}

__global__ void k_flags(uint32_t n, const uint32_t* owner, const Task* tasks, const float4* blo, const float4* bhi,
                        uint32_t* flags) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t t = owner[i];
  flags[i] = t != kNone && goes_left(tasks[t], i, blo[i], bhi[i]) ? 1u : 0u;
}

// Stable partition of every large task's range; primitives of finished
// ranges keep their place.  scan: exclusive prefix sum of the flags.  The
// centroid bounds of the next level's tasks are taken on the way.
__global__ void __launch_bounds__(kLevelThreads)
    k_scatter(uint32_t n, const uint32_t* owner, const Task* tasks, const uint32_t* flags, const uint32_t* scan,
              const uint32_t* ids, const float4* blo, const float4* bhi, uint32_t* ids2, float4* blo2, float4* bhi2,
              uint32_t* owner2, Task* next, BuildCtr* ctr) {
  __shared__ uint32_t sSum[kLevelSlots * 2 * 6], sTask[kLevelSlots];
  uint32_t t[kLevelItems], slot[kLevelItems];
  const uint32_t slots = chunk_slots(n, owner, t, slot, sTask, ctr);
  for (uint32_t j = threadIdx.x; j < slots * 2 * 6; j += kLevelThreads)
    sSum[j] = j % 6 < 3 ? ordered_bits(kInf) : ordered_bits(-kInf);
  __syncthreads();
  for (int e = 0; e < kLevelItems; e++) {
    const uint32_t i = blockIdx.x * kLevelChunk + e * kLevelThreads + threadIdx.x;
    uint32_t key = kNone;
    float c3[3] = {0.f, 0.f, 0.f};
    if (i < n) {
      uint32_t p = i, o = kNone;
      const float4 lo = blo[i], hi = bhi[i];
      if (t[e] != kNone) {
        const Task& tk = tasks[t[e]];
        const uint32_t before = scan[i] - scan[tk.begin];  // left-going primitives of the task before i
        const uint32_t right = flags[i] ? 0u : 1u;
        p = right ? tk.begin + tk.nl + (i - tk.begin - before) : tk.begin + before;
        o = tk.child_task[right];
        if (o != kNone) key = 2 * slot[e] + right;
        const float4 c = centroid(lo, hi);
        c3[0] = c.x, c3[1] = c.y, c3[2] = c.z;
        if (p < tk.begin || p >= tk.end) {  // the bin counts and the flags disagree: report, write nothing
          atomicOr(&ctr->error, 8u);
          p = kNone;
          key = kNone;
        }
      }
      if (p != kNone) {
        ids2[p] = ids[i];
        blo2[p] = lo;
        bhi2[p] = hi;
        owner2[p] = o;
      }
    }
    wave_add<false>(sSum, key, c3, c3);
  }
  __syncthreads();
  for (uint32_t j = threadIdx.x; j < 2 * slots; j += kLevelThreads) {
    const uint32_t* s = sSum + 6 * j;
    const uint32_t c = tasks[sTask[j / 2]].child_task[j % 2];
    if (c == kNone || s[0] > s[3]) continue;
    for (int a = 0; a < 3; a++) {
      atomic_min_f(&next[c].clo[a], from_ordered(s[a]));
      atomic_max_f(&next[c].chi[a], from_ordered(s[3 + a]));
    }
  }
}

// One wave per small task (2 to kSmall = 64 primitives, one per lane): the
// whole subtree, splitting each range at the best SAH position over the
// centroid order of every axis (ties broken by position), with the range
// partitioned stably through LDS.  Ranges of at most max_leaf primitives
// become leaves unless the split is cheaper (the host builder's rule).
constexpr int kSmallWaves = 4;
__global__ void __launch_bounds__(64 * kSmallWaves) k_small(const SmallTask* smalls, uint32_t nSmall, uint32_t* ids,
                                                            float4* blo, float4* bhi, N2* n2, uint32_t maxLeaf) {
  __shared__ float4 sLo[kSmallWaves][kSmall], sHi[kSmallWaves][kSmall];
  __shared__ uint32_t sId[kSmallWaves][kSmall];
  __shared__ uint32_t sStk[kSmallWaves][kSmall][2];  // (node, begin | end << 8)
  const int wave = threadIdx.x >> 6, lane = __lane_id();
  float4* Lo = sLo[wave];
  float4* Hi = sHi[wave];
  uint32_t* Id = sId[wave];
  for (uint32_t t = blockIdx.x * kSmallWaves + wave; t < nSmall; t += gridDim.x * kSmallWaves) {
    const SmallTask st = smalls[t];
    const int m = int(st.end - st.begin);
    if (lane < m) {
      Lo[lane] = blo[st.begin + lane];
      Hi[lane] = bhi[st.begin + lane];
      Id[lane] = ids[st.begin + lane];
    }
    // the subtree's nodes were reserved with the task: an atomic per split on
    // the one node counter bounded this kernel (14.4 ms for 1.3 M splits)
    uint32_t used = 0;
    int sp = 0;
    if (lane == 0) {
      sStk[wave][0][0] = st.node;
      sStk[wave][0][1] = uint32_t(m) << 8;
    }
    sp = 1;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    while (sp > 0) {
      sp--;
      const uint32_t node = __builtin_amdgcn_readfirstlane(sStk[wave][sp][0]);
      const uint32_t be = __builtin_amdgcn_readfirstlane(sStk[wave][sp][1]);
      const int b = int(be & 0xffu), e = int(be >> 8), cnt = e - b;
      const bool act = lane >= b && lane < e;
      const float4 mlo = act ? Lo[lane] : make_float4(kInf, kInf, kInf, 0.f);
      const float4 mhi = act ? Hi[lane] : make_float4(-kInf, -kInf, -kInf, 0.f);
      float nlo[3] = {wave_min(mlo.x), wave_min(mlo.y), wave_min(mlo.z)};
      float nhi[3] = {wave_max(mhi.x), wave_max(mhi.y), wave_max(mhi.z)};
      // candidate: this lane's primitive is the first of the right side in
      // (centroid[a], position) order
      const float4 mc = centroid(mlo, mhi);
      float best = kInf;
      int bestAxis = 0;
      for (int a = 0; a < 3; a++) {
        const float key = comp(mc, a);
        float llo[3] = {kInf, kInf, kInf}, lhi[3] = {-kInf, -kInf, -kInf};
        float rlo[3] = {kInf, kInf, kInf}, rhi[3] = {-kInf, -kInf, -kInf};
        int nl = 0;
        for (int k = b; k < e; k++) {
          const float4 l = Lo[k], h = Hi[k];
          const float ck = comp(centroid(l, h), a);
          const bool left = ck < key || (ck == key && k < lane);
          float* xl = left ? llo : rlo;
          float* xh = left ? lhi : rhi;
          xl[0] = fminf(xl[0], l.x), xl[1] = fminf(xl[1], l.y), xl[2] = fminf(xl[2], l.z);
          xh[0] = fmaxf(xh[0], h.x), xh[1] = fmaxf(xh[1], h.y), xh[2] = fmaxf(xh[2], h.z);
          nl += left ? 1 : 0;
        }
        if (act && nl > 0) {
          const float c = half_area(llo, lhi) * float(nl) + half_area(rlo, rhi) * float(cnt - nl);
          if (c < best) {
            best = c;
            bestAxis = a;
          }
        }
      }
      // wave argmin (lowest lane among equal costs)
      float wc = best;
      int wl = act && best < kInf ? lane : 64;
      for (int o = 32; o > 0; o >>= 1) {
        const float oc = __shfl_xor(wc, o);
        const int ol = __shfl_xor(wl, o);
        if (oc < wc || (oc == wc && ol < wl)) wc = oc, wl = ol;
      }
      // a range of at most max_leaf primitives stays a leaf unless splitting
      // is cheaper: leaf cost n against 1 + SAH cost / parent area
      if (uint32_t(cnt) <= maxLeaf) {
        const float A = half_area(nlo, nhi);
        const float splitCost = A > 0.f && wl < 64 ? 1.f + wc / A : kInf;
        if (cnt <= 1 || float(cnt) <= splitCost) {
          if (lane == 0) {
            N2 leaf;
            for (int a = 0; a < 3; a++) leaf.lo[a] = nlo[a], leaf.hi[a] = nhi[a];
            leaf.left = st.begin + uint32_t(b);
            leaf.count = uint32_t(cnt);
            n2[node] = leaf;
          }
          continue;
        }
      }
      const int winner = wl;
      int axis = 0;
      float wkey = 0.f;
      const bool split_by_key = winner < 64;
      if (split_by_key) {
        axis = __shfl(bestAxis, winner);
        wkey = __shfl(comp(mc, axis), winner);
      }
      // stable partition of [b, e); the left size is counted from the
      // partition itself, so the positions always permute [b, e)
      const float myKey = comp(mc, axis);
      bool left = act && (split_by_key ? (myKey < wkey || (myKey == wkey && lane < winner)) : lane - b < cnt / 2);
      uint64_t lmask = __ballot(left);
      int nlw = __popcll(lmask);
      if (nlw == 0 || nlw == cnt) {  // no usable key split (e.g. NaN centroids): halve the range
        left = act && lane - b < cnt / 2;
        lmask = __ballot(left);
        nlw = __popcll(lmask);
      }
      const uint64_t below = (1ull << lane) - 1ull;
      const uint64_t rmask = __ballot(act && !left);
      const int pos = left ? b + __popcll(lmask & below) : b + nlw + __popcll(rmask & below);
      const uint32_t myId = act ? Id[lane] : 0u;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      if (act) {
        Lo[pos] = mlo;
        Hi[pos] = mhi;
        Id[pos] = myId;
      }
      const uint32_t child = st.nodes + used;
      used += 2;
      if (lane == 0) {
        N2 me;
        for (int a = 0; a < 3; a++) me.lo[a] = nlo[a], me.hi[a] = nhi[a];
        me.left = child;
        me.count = 0;
        n2[node] = me;
        sStk[wave][sp][0] = child;
        sStk[wave][sp][1] = uint32_t(b) | uint32_t(b + nlw) << 8;
        sStk[wave][sp + 1][0] = child + 1;
        sStk[wave][sp + 1][1] = uint32_t(b + nlw) | uint32_t(e) << 8;
      }
      sp += 2;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    if (lane < m) {
      blo[st.begin + lane] = Lo[lane];
      bhi[st.begin + lane] = Hi[lane];
      ids[st.begin + lane] = Id[lane];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

__device__ inline void range_bounds(const float4* blo, const float4* bhi, uint32_t b, uint32_t e, float lo[3], float hi[3]) {
  lo[0] = lo[1] = lo[2] = kInf;
  hi[0] = hi[1] = hi[2] = -kInf;
  for (uint32_t i = b; i < e; i++) {
    float4 l = blo[i], h = bhi[i];
    lo[0] = fminf(lo[0], l.x), lo[1] = fminf(lo[1], l.y), lo[2] = fminf(lo[2], l.z);
    hi[0] = fmaxf(hi[0], h.x), hi[1] = fmaxf(hi[1], h.y), hi[2] = fmaxf(hi[2], h.z);
  }
}

__global__ void k_root_leaf(const float4* blo, const float4* bhi, uint32_t n, N2* n2) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  N2 r;
  range_bounds(blo, bhi, 0, n, r.lo, r.hi);
  r.left = 0;
  r.count = n;
  n2[0] = r;
}

// ---------------------------------------------------------------- collapse to 4-wide nodes
struct Job {
  uint32_t n2, n4;
};

__device__ __forceinline__ float widen(float v, bool up) {
  float m = fabsf(v) * 4.0f * 1.1920929e-7f + 1e-30f;
  return up ? v + m : v - m;
}

__global__ void k_collapse(const Job* jobs, uint32_t nJobs, const N2* n2, BvhNode4* out, Job* next, uint32_t* ctr) {
  uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= nJobs) return;
  Job jb = jobs[j];
  uint32_t kid[4];
  int nk = 0;
  const N2 x = n2[jb.n2];
  if (x.count > 0) {
    kid[nk++] = jb.n2;
  } else {
    kid[nk++] = x.left;
    kid[nk++] = x.left + 1;
  }
  while (nk < 4) {
    int bi = -1;
    float ba = -1.f;
    for (int k = 0; k < nk; k++) {
      const N2& c = n2[kid[k]];
      if (c.count > 0) continue;
      float a = half_area(c.lo, c.hi);
      if (a > ba) {
        ba = a;
        bi = k;
      }
    }
    if (bi < 0) break;
    uint32_t l = n2[kid[bi]].left;
    kid[bi] = l;
    kid[nk++] = l + 1;
  }
  // the node's inner children get consecutive ids, so siblings share cache lines
  int inner = 0;
  for (int s = 0; s < nk; s++) inner += n2[kid[s]].count > 0 ? 0 : 1;
  uint32_t base = 0, qbase = 0;
  if (inner) {
    base = atomicAdd(&ctr[0], uint32_t(inner));
    qbase = atomicAdd(&ctr[1], uint32_t(inner));
  }
  BvhNode4 o;
  for (int s = 0; s < 4; s++) {
    if (s >= nk) {
      o.lox[s] = o.loy[s] = o.loz[s] = kInf;
      o.hix[s] = o.hiy[s] = o.hiz[s] = -kInf;
      o.child[s] = -1;
      o.count[s] = 0;
      continue;
    }
    const N2 c = n2[kid[s]];
    o.lox[s] = widen(c.lo[0], false);
    o.loy[s] = widen(c.lo[1], false);
    o.loz[s] = widen(c.lo[2], false);
    o.hix[s] = widen(c.hi[0], true);
    o.hiy[s] = widen(c.hi[1], true);
    o.hiz[s] = widen(c.hi[2], true);
    if (c.count > 0) {
      o.child[s] = int32_t(c.left);
      o.count[s] = c.count;
    } else {
      next[qbase] = Job{kid[s], base};
      o.child[s] = int32_t(base);
      o.count[s] = 0;
      base++;
      qbase++;
    }
  }
  out[jb.n4] = o;
}

// Worst-case traversal stack entries of the nodes [begin, end) of one level,
// from those of the next level (launched deepest level first).
__global__ void k_stack_need(const BvhNode4* nodes, uint32_t begin, uint32_t end, uint32_t* need) {
  const uint32_t i = begin + blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= end) return;
  const BvhNode4& nd = nodes[i];
  uint32_t inner = 0, deepest = 0;
  for (int s = 0; s < 4; s++)
    if (nd.child[s] >= 0 && nd.count[s] == 0) {
      inner++;
      deepest = max(deepest, need[nd.child[s]]);
    }
  need[i] = inner ? inner - 1 + deepest : 0u;
}

__global__ void k_gather_prims(const float4* rec, const uint32_t* ids, uint32_t n, float4* out) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float4* s = rec + 3 * size_t(ids[i]);
  out[3 * size_t(i)] = s[0];
  out[3 * size_t(i) + 1] = s[1];
  out[3 * size_t(i) + 2] = s[2];
}

// SAH cost (traversal 1, intersection 1, relative to the root area).
__global__ void k_sah(const BvhNode4* nodes, uint32_t m, float rootA, double* cost) {
  double c = 0.0;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < m; i += gridDim.x * blockDim.x) {
    const BvhNode4& nd = nodes[i];
    for (int s = 0; s < 4; s++) {
      if (nd.child[s] < 0) continue;
      float lo[3] = {nd.lox[s], nd.loy[s], nd.loz[s]}, hi[3] = {nd.hix[s], nd.hiy[s], nd.hiz[s]};
      float a = 2.f * half_area(lo, hi) / rootA;
      c += nd.count[s] > 0 ? a * float(nd.count[s]) : a;
    }
  }
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
  if (__lane_id() == 0 && c != 0.0) atomicAdd(cost, c);
}

// ---------------------------------------------------------------- traversal nodes
// One thread per node of a level (bvh_wide.h).  EMIT = false: sums[j] =
// wide_count.  EMIT = true, after an exclusive scan of the sums: wide_emit.
struct WideLevel {
  uint32_t nodes, next, prims;  // first node of this level, of the next level, first primitive this level places
};
template <bool EMIT>
__global__ void __launch_bounds__(64) k_wide(const WideJob* jobs, uint32_t nJobs, BvhNode4* nodes, unsigned long long* sums, WideKids* kids,
                       WideLevel lv, BvhNode8* out, WideJob* next, uint32_t* perm, uint32_t* error) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= nJobs) {
    if (!EMIT && j == nJobs) sums[j] = 0ull;  // the scan's last entry is the level's total
    return;
  }
  const WideJob jb = jobs[j];
  if (!EMIT) {
    sums[j] = wide_count(nodes, jb, kids[j]);
    return;
  }
  const uint32_t inner = uint32_t(sums[j]), prims = uint32_t(sums[j] >> 32);
  if (!wide_emit(nodes, jb, kids[j], lv.next + inner, jb.mask & kWideRest ? jb.begin : lv.prims + prims, out + lv.nodes + j,
                 next + inner, perm))
    atomicOr(error, 1u);
}

// All levels of a small tree in one block: a level of k_wide costs two launches,
// a scan and a wait for its size, whatever the number of its nodes.  The jobs
// of a level are taken in groups of kWideThreads with running sums, so the
// nodes are those of the level passes.  Bound, as k_wide, by the latency of one
// thread's steps, here on one compute unit.  Whole builds, level passes / one
// block: 82 nodes of the 4-wide tree 1321 / 1251 us, 1611 2408 / 2302, 3651
// 2897 / 2862, 8720 3123 / 3501.
constexpr int kWideThreads = 512;
constexpr uint32_t kWideTreeNodes = 4096;  // largest 4-wide tree made so
struct WideTotals {
  uint32_t nodes, prims, error;  // error: 1 a box cannot be bounded, 2 the buffers are exceeded
};
__global__ void __launch_bounds__(kWideThreads) k_wide_tree(WideJob* cur, WideJob* nxt, BvhNode4* nodes, WideKids* kids, uint32_t cap,
                                                            uint32_t n, BvhNode8* out, uint32_t* perm, WideTotals* totals) {
  constexpr int kWaves = kWideThreads / 64;
  __shared__ unsigned long long sWave[kWaves];
  __shared__ uint32_t sBad;
  const uint32_t lane = __lane_id(), wave = threadIdx.x >> 6;
  if (threadIdx.x == 0) {
    cur[0] = WideJob{0, kWideAll, 0, 0};
    sBad = 0;
  }
  __syncthreads();
  uint32_t jobs = 1, first = 0, prims = 0;  // of this level
  while (jobs > 0) {
    const uint32_t next = first + jobs;
    unsigned long long base = 0;  // inner children (low word) and primitives (high word) of the groups before
    for (uint32_t g = 0; g < jobs; g += kWideThreads) {
      const uint32_t j = g + threadIdx.x;
      const bool mine = j < jobs;
      WideJob jb{};
      unsigned long long mySum = 0;
      if (mine) {
        jb = cur[j];
        mySum = wide_count(nodes, jb, kids[j]);
      }
      unsigned long long incl = mySum;
      for (int o = 1; o < 64; o <<= 1) {
        const unsigned long long v = __shfl_up(incl, o);
        if (lane >= uint32_t(o)) incl += v;
      }
      if (lane == 63) sWave[wave] = incl;
      __syncthreads();
      unsigned long long before = base, total = 0;
      for (int w = 0; w < kWaves; w++) {
        before += uint32_t(w) < wave ? sWave[w] : 0ull;
        total += sWave[w];
      }
      before += incl - mySum;
      base += total;
      if (uint64_t(next) + uint32_t(base) > cap || uint32_t(base >> 32) > n - prims) {  // the same in every thread
        if (threadIdx.x == 0) *totals = WideTotals{0, 0, 2};
        return;
      }
      if (mine) {
        const uint32_t inner = uint32_t(before);
        if (!wide_emit(nodes, jb, kids[j], next + inner, jb.mask & kWideRest ? jb.begin : prims + uint32_t(before >> 32),
                       out + first + j, nxt + inner, perm))
          sBad = 1;
      }
      __syncthreads();  // sWave is read; the next level's jobs are written
    }
    first = next;
    jobs = uint32_t(base);
    prims += uint32_t(base >> 32);
    WideJob* t = cur;
    cur = nxt;
    nxt = t;
  }
  if (threadIdx.x == 0) *totals = WideTotals{first, prims, sBad};
}

unsigned Grid(uint64_t n, unsigned t = 256) { return unsigned((n + t - 1) / t); }

}  // namespace

// Consecutive arrays in one allocation; with base == nullptr it only measures.
struct Carver {
  char* base;
  size_t used = 0;
  template <class T>
  T* take(size_t n) {
    T* r = reinterpret_cast<T*>(base ? base + used : nullptr);
    used += (n * sizeof(T) + 255) & ~size_t(255);
    return r;
  }
};

uint32_t BuildWideNodes(DeviceBuffer& nodes, uint32_t m, uint32_t maxLeaf, DeviceBuffer& prims, uint32_t n, hipStream_t st,
                        DeviceBuffer& work, DeviceBuffer& out) {
  // One node per BvhNode4 at most, unless its leaves hold more than
  // kWideNodePrims (four of at most a quarter of that never do): a chain then has
  // at most one node per leaf, one more per kWideNodePrims and one for the rest.
  const size_t cap = maxLeaf <= kWideNodePrims / 4 ? size_t(m) : 5 * size_t(m) + n / kWideNodePrims + 8;
  size_t scanBytes = 0;
  HipCheck(hipcub::DeviceScan::ExclusiveSum(nullptr, scanBytes, static_cast<unsigned long long*>(nullptr),
                                            static_cast<unsigned long long*>(nullptr), int(cap + 1), st),
           "wide scan size");
  BvhNode8* wide;
  WideJob *cur, *nxt;
  unsigned long long* sums;
  WideKids* kids;
  float4* ordered;
  uint32_t *perm, *flag;
  WideTotals* totals;
  char* tmp;
  const auto carve = [&](Carver c) {
    wide = c.take<BvhNode8>(cap);
    cur = c.take<WideJob>(cap);
    nxt = c.take<WideJob>(cap);
    sums = c.take<unsigned long long>(cap + 1);
    kids = c.take<WideKids>(cap);
    perm = c.take<uint32_t>(std::max(n, 1u));
    ordered = c.take<float4>(3 * size_t(std::max(n, 1u)));
    flag = c.take<uint32_t>(1);
    totals = c.take<WideTotals>(1);
    tmp = c.take<char>(std::max<size_t>(scanBytes, 16));
    return c.used;
  };
  const size_t need = carve(Carver{nullptr});
  if (work.bytes < need) work.alloc(need);
  carve(Carver{static_cast<char*>(work.ptr)});
  uint32_t e = 0;
  WideLevel lv{0, 1, 0};
  if (m <= kWideTreeNodes) {
    hipLaunchKernelGGL(k_wide_tree, dim3(1), dim3(kWideThreads), 0, st, cur, nxt, nodes.as<BvhNode4>(), kids, uint32_t(cap), n, wide,
                       perm, totals);
    WideTotals t{};
    HipCheck(hipMemcpyAsync(&t, totals, sizeof(t), hipMemcpyDeviceToHost, st), "wide nodes");
    HipCheck(hipStreamSynchronize(st), "wide nodes");
    if (t.error == 2) throw std::runtime_error("traversal nodes exceed their buffers");
    lv.nodes = t.nodes;
    lv.prims = t.prims;
    e = t.error;
  } else {
    HipCheck(hipMemsetAsync(flag, 0, 4, st), "wide node flag");
    const WideJob root{0, kWideAll, 0, 0};
    HipCheck(hipMemcpyAsync(cur, &root, sizeof(root), hipMemcpyHostToDevice, st), "wide root");
    uint32_t nJobs = 1;
    while (nJobs > 0) {
      hipLaunchKernelGGL(k_wide<false>, dim3(Grid(nJobs + 1, 64)), dim3(64), 0, st, cur, nJobs, nodes.as<BvhNode4>(), sums, kids, lv,
                         nullptr, nullptr, nullptr, nullptr);
      size_t bytes = scanBytes;
      HipCheck(hipcub::DeviceScan::ExclusiveSum(tmp, bytes, sums, sums, int(nJobs + 1), st), "wide scan");
      unsigned long long total = 0;
      HipCheck(hipMemcpyAsync(&total, sums + nJobs, 8, hipMemcpyDeviceToHost, st), "wide level");
      HipCheck(hipStreamSynchronize(st), "wide level");
      const uint32_t inner = uint32_t(total), placed = uint32_t(total >> 32);
      lv.next = lv.nodes + nJobs;
      if (placed > n - lv.prims || size_t(lv.next) + inner > cap)
        throw std::runtime_error("traversal nodes exceed their buffers");
      hipLaunchKernelGGL(k_wide<true>, dim3(Grid(nJobs, 64)), dim3(64), 0, st, cur, nJobs, nodes.as<BvhNode4>(), sums, kids, lv, wide,
                         nxt, perm, flag);
      lv.nodes = lv.next;
      lv.prims += placed;
      nJobs = inner;
      std::swap(cur, nxt);
    }
    HipCheck(hipMemcpyAsync(&e, flag, 4, hipMemcpyDeviceToHost, st), "wide node flag");
    HipCheck(hipStreamSynchronize(st), "wide nodes");
  }
  if (e) throw std::runtime_error("BVH node bounds cannot be quantised (non-finite boxes?)");
  if (lv.prims != n) throw std::runtime_error("traversal nodes do not reference every primitive");
  out.alloc(size_t(lv.nodes) * sizeof(BvhNode8));
  HipCheck(hipMemcpyAsync(out.ptr, wide, size_t(lv.nodes) * sizeof(BvhNode8), hipMemcpyDeviceToDevice, st), "wide nodes");
  if (n) {
    hipLaunchKernelGGL(k_gather_prims, dim3(Grid(n)), dim3(256), 0, st, prims.as<float4>(), perm, n, ordered);
    HipCheck(hipMemcpyAsync(prims.ptr, ordered, size_t(n) * 48, hipMemcpyDeviceToDevice, st), "ordered primitives");
  }
  HipCheck(hipStreamSynchronize(st), "wide nodes");
  return lv.nodes;
}

void BuildBvh4Device(const PrimSource& src, int maxLeaf, hipStream_t st, DeviceBuffer& nodesOut, DeviceBuffer& primsOut,
                     bool& outputsValid, DeviceBuffer& work, DeviceBvhStats& stats) {
  const uint32_t n = src.count;
  if (n == 0) throw std::runtime_error("scene has no primitives");
  if (maxLeaf < 1 || maxLeaf > 16) throw std::runtime_error("max_leaf_size must lie in [1, 16]");
  auto t0 = std::chrono::steady_clock::now();
  const uint32_t maxNodes = 2 * n;
  const uint32_t maxTasks = n / (kSmall + 1) + 2;
  const uint32_t maxSmall = n / 2 + 2;  // small tasks hold at least two primitives
  const uint32_t others = uint32_t(src.other_rec.size() / 3);
  size_t sortBytes = 0, scanBytes = 0;
  HipCheck(hipcub::DeviceRadixSort::SortPairs(nullptr, sortBytes, static_cast<uint64_t*>(nullptr), static_cast<uint64_t*>(nullptr),
                                              static_cast<uint32_t*>(nullptr), static_cast<uint32_t*>(nullptr), int(n), 0, 63, st),
           "radix sort size");
  HipCheck(hipcub::DeviceScan::ExclusiveSum(nullptr, scanBytes, static_cast<uint32_t*>(nullptr),
                                            static_cast<uint32_t*>(nullptr), int(n), st),
           "scan size");
  // One allocation: what lives to the end, then the arrays of the binary build
  // and, in their place afterwards, those of the collapse (a 4-wide node per
  // inner binary node at most).
  float4 *rec, *lo, *hi, *lo2, *hi2, *otherRec;
  float *box, *cb, *otherBox;
  uint64_t *keys, *keys2;
  uint32_t *ids0, *ids, *ids2, *own, *own2, *flags, *scan, *jc, *need;
  N2* n2;
  BuildCtr* ctr;
  Task *cur, *nxt;
  SmallTask* smalls;
  Bin* bins;
  PrimSegment* segs;
  double* cost;
  char* tmp;
  BvhNode4* nodes;
  Job *jcur, *jnxt;
  const auto carve = [&](Carver c) {
    rec = c.take<float4>(3 * size_t(n));
    n2 = c.take<N2>(maxNodes);
    ids0 = c.take<uint32_t>(n);
    ids = c.take<uint32_t>(n);
    ids2 = c.take<uint32_t>(n);
    ctr = c.take<BuildCtr>(1);
    jc = c.take<uint32_t>(2);
    cost = c.take<double>(1);
    Carver d = c;
    box = c.take<float>(6 * size_t(n));
    cb = c.take<float>(6);
    keys = c.take<uint64_t>(n);
    keys2 = c.take<uint64_t>(n);
    lo = c.take<float4>(n);
    hi = c.take<float4>(n);
    lo2 = c.take<float4>(n);
    hi2 = c.take<float4>(n);
    own = c.take<uint32_t>(n);
    own2 = c.take<uint32_t>(n);
    flags = c.take<uint32_t>(n);
    scan = c.take<uint32_t>(n);
    cur = c.take<Task>(maxTasks);
    nxt = c.take<Task>(maxTasks);
    smalls = c.take<SmallTask>(maxSmall);
    bins = c.take<Bin>(size_t(maxTasks) * 3 * kBins);
    tmp = c.take<char>(std::max<size_t>(std::max(sortBytes, scanBytes), 16));
    segs = c.take<PrimSegment>(src.segs.size());
    otherRec = c.take<float4>(std::max(3 * size_t(others), size_t(1)));
    otherBox = c.take<float>(std::max(6 * size_t(others), size_t(1)));
    nodes = d.take<BvhNode4>(n);
    jcur = d.take<Job>(n);
    jnxt = d.take<Job>(n);
    need = d.take<uint32_t>(n);
    return std::max(c.used, d.used);
  };
  work.alloc(carve(Carver{nullptr}));
  carve(Carver{static_cast<char*>(work.ptr)});
  // primitives
  HipCheck(hipMemcpyAsync(segs, src.segs.data(), src.segs.size() * sizeof(PrimSegment), hipMemcpyHostToDevice, st), "segments");
  if (others) {
    HipCheck(hipMemcpyAsync(otherRec, src.other_rec.data(), size_t(others) * 48, hipMemcpyHostToDevice, st), "primitives");
    HipCheck(hipMemcpyAsync(otherBox, src.other_box.data(), size_t(others) * 24, hipMemcpyHostToDevice, st), "bounds");
  }
  hipLaunchKernelGGL(k_primitives, dim3(Grid(n)), dim3(256), 0, st, segs, uint32_t(src.segs.size()), src.d_tris, otherRec,
                     otherBox, n, rec, box);
  // ordering
  const float init[6] = {kInf, kInf, kInf, -kInf, -kInf, -kInf};
  HipCheck(hipMemcpyAsync(cb, init, 24, hipMemcpyHostToDevice, st), "centroid init");
  hipLaunchKernelGGL(k_centroid_bounds, dim3(std::min(Grid(n), 256u)), dim3(256), 0, st, box, n, cb);
  hipLaunchKernelGGL(k_morton, dim3(Grid(n)), dim3(256), 0, st, box, n, cb, keys, ids0);
  HipCheck(hipcub::DeviceRadixSort::SortPairs(tmp, sortBytes, keys, keys2, ids0, ids, int(n), 0, 63, st), "radix sort");
  hipLaunchKernelGGL(k_gather_bounds, dim3(Grid(n)), dim3(256), 0, st, box, ids, n, lo, hi);
  // top-down levels
  const Caps caps{maxNodes, maxTasks, maxSmall};
  uint32_t levels = 0, nSmall = 0;
  BuildCtr c0{1, 0, 0, 0};
  if (n == 1) {
    hipLaunchKernelGGL(k_root_leaf, dim3(1), dim3(64), 0, st, lo, hi, n, n2);
  } else if (n <= kSmall) {
    const SmallTask root{0, 0, n, 1};
    HipCheck(hipMemcpyAsync(smalls, &root, sizeof(root), hipMemcpyHostToDevice, st), "root task");
    c0.nodes = 1 + 2 * (n - 1);
    c0.smalls = 1;
    nSmall = 1;
  } else {
    Task root{};
    root.node = 0;
    root.begin = 0;
    root.end = n;
    root.axis = 3;
    root.child_task[0] = root.child_task[1] = kNone;
    HipCheck(hipMemcpyAsync(&root.clo, cb, 12, hipMemcpyDeviceToHost, st), "centroid bounds");
    HipCheck(hipMemcpyAsync(&root.chi, cb + 3, 12, hipMemcpyDeviceToHost, st), "centroid bounds");
    HipCheck(hipStreamSynchronize(st), "centroid bounds");
    HipCheck(hipMemcpyAsync(cur, &root, sizeof(Task), hipMemcpyHostToDevice, st), "root task");
    HipCheck(hipMemsetAsync(own, 0, size_t(n) * 4, st), "owners");
  }
  HipCheck(hipMemcpyAsync(ctr, &c0, sizeof(c0), hipMemcpyHostToDevice, st), "counters");
  if (n > kSmall) {
    uint32_t nTasks = 1;
    while (nTasks > 0) {
      if (++levels > 128) throw std::runtime_error("BVH build did not converge");
      hipLaunchKernelGGL(k_bins_clear, dim3(Grid(uint64_t(nTasks) * 3 * kBins)), dim3(256), 0, st, bins, nTasks * 3 * kBins);
      hipLaunchKernelGGL(k_bins_accum, dim3(Grid(n, kLevelChunk)), dim3(kLevelThreads), 0, st, n, own, cur, lo, hi, bins, ctr);
      HipCheck(hipMemsetAsync(&ctr->tasks, 0, 4, st), "level counter");
      hipLaunchKernelGGL(k_split, dim3(Grid(nTasks, kSplitWaves)), dim3(64 * kSplitWaves), 0, st, cur, nTasks, bins, n2, nxt, smalls, ctr, caps);
      hipLaunchKernelGGL(k_flags, dim3(Grid(n)), dim3(256), 0, st, n, own, cur, lo, hi, flags);
      size_t bytes = scanBytes;
      HipCheck(hipcub::DeviceScan::ExclusiveSum(tmp, bytes, flags, scan, int(n), st), "flag scan");
      hipLaunchKernelGGL(k_scatter, dim3(Grid(n, kLevelChunk)), dim3(kLevelThreads), 0, st, n, own, cur, flags, scan, ids, lo, hi,
                         ids2, lo2, hi2, own2, nxt, ctr);
      std::swap(ids, ids2);
      std::swap(lo, lo2);
      std::swap(hi, hi2);
      std::swap(own, own2);
      BuildCtr h{};
      HipCheck(hipMemcpyAsync(&h, ctr, sizeof(h), hipMemcpyDeviceToHost, st), "level readback");
      HipCheck(hipStreamSynchronize(st), "BVH level");
      if (h.error || h.nodes > maxNodes || h.tasks > maxTasks || h.smalls > maxSmall)
        throw std::runtime_error("BVH build exceeded its buffers");
      nTasks = h.tasks;
      nSmall = h.smalls;
      std::swap(cur, nxt);
    }
  }
  if (nSmall) {
    const uint32_t blocks = std::min<uint32_t>((nSmall + kSmallWaves - 1) / kSmallWaves, 65535u * 4u);
    hipLaunchKernelGGL(k_small, dim3(blocks), dim3(64 * kSmallWaves), 0, st, smalls, nSmall, ids, lo, hi, n2, uint32_t(maxLeaf));
  }
  // collapse
  const Job rj{0, 0};
  HipCheck(hipMemcpyAsync(jcur, &rj, sizeof(rj), hipMemcpyHostToDevice, st), "root job");
  uint32_t hjc[2] = {1, 0};
  uint32_t nJobs = 1, depth = 0;
  std::vector<uint32_t> levelStart{0u};  // the nodes of level k are [levelStart[k], levelStart[k + 1])
  while (nJobs > 0) {
    depth++;
    levelStart.push_back(hjc[0]);
    hjc[1] = 0;
    HipCheck(hipMemcpyAsync(jc, hjc, 8, hipMemcpyHostToDevice, st), "collapse counters");
    hipLaunchKernelGGL(k_collapse, dim3(Grid(nJobs, 64)), dim3(64), 0, st, jcur, nJobs, n2, nodes, jnxt, jc);
    HipCheck(hipMemcpyAsync(hjc, jc, 8, hipMemcpyDeviceToHost, st), "collapse readback");
    HipCheck(hipStreamSynchronize(st), "collapse level");
    nJobs = hjc[1];
    std::swap(jcur, jnxt);
  }
  const uint32_t n4 = hjc[0];
  levelStart.push_back(n4);
  for (size_t k = levelStart.size() - 1; k-- > 0;) {
    const uint32_t b = levelStart[k], e = levelStart[k + 1];
    if (e > b) hipLaunchKernelGGL(k_stack_need, dim3(Grid(e - b)), dim3(256), 0, st, nodes, b, e, need);
  }
  uint32_t stackNeed = 0;
  HipCheck(hipMemcpyAsync(&stackNeed, need, sizeof(uint32_t), hipMemcpyDeviceToHost, st), "stack need");
  outputsValid = false;
  nodesOut.alloc(size_t(n4) * sizeof(BvhNode4));
  HipCheck(hipMemcpyAsync(nodesOut.ptr, nodes, size_t(n4) * sizeof(BvhNode4), hipMemcpyDeviceToDevice, st), "nodes");
  primsOut.alloc(size_t(n) * 48);
  hipLaunchKernelGGL(k_gather_prims, dim3(Grid(n)), dim3(256), 0, st, rec, ids, n, primsOut.as<float4>());
  // statistics: SAH cost relative to the root box
  BvhNode4 root;
  HipCheck(hipMemcpyAsync(&root, nodes, sizeof(root), hipMemcpyDeviceToHost, st), "root readback");
  HipCheck(hipStreamSynchronize(st), "BVH finish");
  float rlo[3] = {kInf, kInf, kInf}, rhi[3] = {-kInf, -kInf, -kInf};
  for (int s = 0; s < 4; s++) {
    if (root.child[s] < 0) continue;
    rlo[0] = std::min(rlo[0], root.lox[s]), rlo[1] = std::min(rlo[1], root.loy[s]), rlo[2] = std::min(rlo[2], root.loz[s]);
    rhi[0] = std::max(rhi[0], root.hix[s]), rhi[1] = std::max(rhi[1], root.hiy[s]), rhi[2] = std::max(rhi[2], root.hiz[s]);
  }
  float dx = rhi[0] - rlo[0], dy = rhi[1] - rlo[1], dz = rhi[2] - rlo[2];
  float rootA = 2.f * (dx * dy + dy * dz + dz * dx);
  double sah = 1.0;
  if (rootA > 0.f) {
    HipCheck(hipMemsetAsync(cost, 0, 8, st), "sah");
    hipLaunchKernelGGL(k_sah, dim3(std::min(Grid(n4), 256u)), dim3(256), 0, st, nodes, n4, rootA, cost);
    double c = 0;
    HipCheck(hipMemcpyAsync(&c, cost, 8, hipMemcpyDeviceToHost, st), "sah readback");
    HipCheck(hipStreamSynchronize(st), "sah");
    sah += c;
  }
  HipCheck(hipGetLastError(), "BVH kernels");
  stats.node_count = n4;
  stats.depth = depth;
  stats.stack_need = stackNeed;
  stats.levels = levels;
  stats.sah_cost = float(sah);
  stats.build_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
}

}  // namespace rad
