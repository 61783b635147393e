// Device ray traversal over the 8-wide quantised BVH: closest hit
// (Embree::RayIntersectPreliminary, embree.cpp:87-111) and occlusion
// (Embree::RayIntersect, embree.cpp:79-85).
#pragma once

#include "scene_dev.h"

namespace rad {

struct Hit {
  float t, u, v;
  uint32_t prim;
  uint32_t geom;  // 0xffffffff = miss
};

// Products of the primitive tests with every rounding spelled out (explicit
// fused multiply-adds in a fixed association), so the device and the host
// oracle produce bit-identical t, u, v whatever contraction the compiler
// applies elsewhere.
__device__ __forceinline__ float dotx(f3 a, f3 b) { return fmaf(a.x, b.x, fmaf(a.y, b.y, a.z * b.z)); }
__device__ __forceinline__ f3 crossx(f3 a, f3 b) {
  return mk(fmaf(a.y, b.z, -(a.z * b.y)), fmaf(a.z, b.x, -(a.x * b.z)), fmaf(a.x, b.y, -(a.y * b.x)));
}

// Moller-Trumbore in the form Embree 3 applies to its TriangleM primitives:
// e1 = v0 - v1, e2 = v2 - v0, Ng = e2 x e1, C = v0 - O, R = C x D,
// accept den != 0, U, V >= 0, U + V <= |den|, |den|*tnear < T <= |den|*tfar.
// Traversal keeps only t = T / |den| of the closest hit; tri_uv recomputes
// U, V and |den| with the same operations once the ray is finished.
__device__ __forceinline__ bool isect_tri(f3 v0, f3 v1, f3 v2, f3 o, f3 d, float tnear, float tfar, float& t) {
  f3 e1 = v0 - v1;
  f3 e2 = v2 - v0;
  f3 ng = crossx(e2, e1);
  f3 c = v0 - o;
  f3 r = crossx(c, d);
  float den = dotx(ng, d);
  float absDen = fabsf(den);
  float U = dotx(r, e2);
  float V = dotx(r, e1);
  if (den < 0.f) {
    U = -U;
    V = -V;
  }
  if (!(den != 0.f && U >= 0.f && V >= 0.f && U + V <= absDen)) return false;
  float T = dotx(ng, c);
  if (den < 0.f) T = -T;
  if (!(absDen * tnear < T && T <= absDen * tfar)) return false;
  t = T / absDen;
  return true;
}

__device__ __forceinline__ void tri_uv(f3 v0, f3 v1, f3 v2, f3 o, f3 d, float& u, float& v) {
  f3 e1 = v0 - v1;
  f3 e2 = v2 - v0;
  f3 ng = crossx(e2, e1);
  f3 c = v0 - o;
  f3 r = crossx(c, d);
  float den = dotx(ng, d);
  float absDen = fabsf(den);
  float U = dotx(r, e2);
  float V = dotx(r, e1);
  if (den < 0.f) {
    U = -U;
    V = -V;
  }
  u = U / absDen;
  v = V / absDen;
}

// Sphere user geometry (sphere.cpp:40-54 with SolveQuadratic, math_ext.h:79-97).
__device__ __forceinline__ bool isect_sphere(f3 center, float radius, f3 ro, f3 rd, float near, float far, float& t) {
  f3 o = ro - center;
  float a = dotx(rd, rd);
  float b = 2.0f * dotx(o, rd);
  float c = fmaf(-radius, radius, dotx(o, o));
  bool linearCase = a == 0.0f;
  bool validLinear = linearCase && b != 0.0f;
  float x0 = -c / b, x1 = -c / b;
  float discrim = fmaf(b, b, -((4.0f * a) * c));
  bool validQuadratic = !linearCase && (discrim >= 0.0f);
  if (validQuadratic) {
    float rootDiscrim = sqrtf(discrim);
    float temp = -0.5f * (b + copysignf(rootDiscrim, b));
    float x0p = temp / a;
    float x1p = c / temp;
    float x0m = fminf(x0p, x1p);
    float x1m = fmaxf(x0p, x1p);
    x0 = linearCase ? x0 : x0m;
    x1 = linearCase ? x0 : x1m;
  }
  bool found = validLinear || validQuadratic;
  bool outBounds = !(x0 <= far && x1 >= near);
  bool inBounds = x0 < near && x1 > far;
  if (!(found && !outBounds && !inBounds)) return false;
  t = x0 < 0.f ? x1 : x0;
  return true;
}

// Rectangle user geometry (rectangle.cpp:34-46): object-space plane z = 0,
// |x|, |y| <= 1, with an unnormalised object-space direction.
__device__ __forceinline__ bool isect_rect(const Affine& toObj, f3 ro, f3 rd, float near, float far, float& t,
                                           float& u, float& v) {  // u, v: the local hit point
  const float* m = toObj.m;
  f3 o = mk(fmaf(m[0], ro.x, fmaf(m[1], ro.y, fmaf(m[2], ro.z, m[3]))),
            fmaf(m[4], ro.x, fmaf(m[5], ro.y, fmaf(m[6], ro.z, m[7]))),
            fmaf(m[8], ro.x, fmaf(m[9], ro.y, fmaf(m[10], ro.z, m[11]))));
  f3 d = mk(fmaf(m[0], rd.x, fmaf(m[1], rd.y, m[2] * rd.z)), fmaf(m[4], rd.x, fmaf(m[5], rd.y, m[6] * rd.z)),
            fmaf(m[8], rd.x, fmaf(m[9], rd.y, m[10] * rd.z)));
  float tt = -o.z / d.z;
  f3 local = mk(fmaf(d.x, tt, o.x), fmaf(d.y, tt, o.y), fmaf(d.z, tt, o.z));
  if (!(tt >= near && tt <= far && fabsf(local.x) <= 1.f && fabsf(local.y) <= 1.f)) return false;
  t = tt;
  u = local.x;
  v = local.y;
  return true;
}

__device__ __forceinline__ f3 xyz(float4 a) { return mk(a.x, a.y, a.z); }

// Test one primitive record (its three float4, already loaded) against the
// segment (tnear, tfar]; on a hit `tfar` becomes its distance.
__device__ __forceinline__ bool isect_rec(const DevScene& s, float4 a, float4 b, float4 c, f3 o, f3 d, float tnear,
                                          float& tfar) {
  const uint32_t kind = __float_as_uint(c.w);
  float t;
  if (kind == PRIM_TRI) {
    if (!isect_tri(xyz(a), xyz(b), xyz(c), o, d, tnear, tfar, t)) return false;
  } else if (kind == PRIM_SPHERE) {
    if (!isect_sphere(xyz(a), a.w, o, d, tnear, tfar, t)) return false;
  } else {
    float u, v;
    if (!isect_rect(s.shapes[__float_as_uint(b.w)].to_local, o, d, tnear, tfar, t, u, v)) return false;
  }
  tfar = t;
  return true;
}
__device__ __forceinline__ bool isect_prim(const DevScene& s, uint32_t p, f3 o, f3 d, float tnear, float& tfar) {
  const float4* rec = s.prims + 3 * size_t(p);
  return isect_rec(s, rec[0], rec[1], rec[2], o, d, tnear, tfar);
}

// The hit record of primitive p at distance t (the closest hit the
// traversal kept): geometry and primitive ids from the record, u, v
// recomputed with the arithmetic of the test that accepted it.
__device__ __forceinline__ void prim_hit(const DevScene& s, uint32_t p, f3 o, f3 d, float t, Hit& h) {
  const float4* rec = s.prims + 3 * size_t(p);
  const float4 a = rec[0], b = rec[1], c = rec[2];
  const uint32_t kind = __float_as_uint(c.w);
  h.t = t;
  h.u = 0.f;
  h.v = 0.f;
  if (kind == PRIM_TRI) {
    tri_uv(xyz(a), xyz(b), xyz(c), o, d, h.u, h.v);
    h.geom = __float_as_uint(a.w);
    h.prim = __float_as_uint(b.w);
  } else if (kind == PRIM_SPHERE) {
    h.geom = __float_as_uint(b.w);
    h.prim = 0;
  } else {
    const uint32_t g = __float_as_uint(b.w);
    float tt;
    isect_rect(s.shapes[g].to_local, o, d, -kInf, kInf, tt, h.u, h.v);
    h.geom = g;
    h.prim = 0;
  }
}

// ---------------------------------------------------------------- traversal
// A ray walks groups of siblings: the inner children of one node that it hits
// are one group (first child's index, hit mask in visiting order, the node's
// inner mask), the current group is in registers, and a node whose own group
// replaces an unfinished one pushes that one: at most one push per node, and
// none for the children themselves.  Each lane keeps the newest kLdsStack
// entries in LDS (a ring, lane-interleaved so a wave's accesses are
// conflict-free), older ones in a private overflow array that only deep
// traversals touch.
constexpr int kStackDepth = int(kGroupStackEntries);
constexpr int kLdsStack = 4;
constexpr int kTraceBlock = 256;  // threads per block of every traversal kernel

// LDS pointers spelled with their address space, so accesses compile to
// ds_read / ds_write rather than flat accesses.
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) u32x2 lds_u2;
typedef __attribute__((address_space(3))) u32x4 lds_u4;
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef __attribute__((address_space(3))) float lds_f32;
typedef __attribute__((address_space(3))) unsigned long long lds_u64;

// Per-lane private overflow of a traversal stack (entries below the LDS ring).
struct TraceOverflow {
  uint2 e[kStackDepth - kLdsStack];
};

// The struct holds no arrays, so its fields stay in registers; only the
// overflow array, indexed by the stack depth, lives in private memory.
struct TraceStack {
  lds_u64* ring;  // entry k of this lane at ring[k * kTraceBlock]
  uint2* ov;      // TraceOverflow of this lane
  int sp, lo;     // entries [0, lo) live in the overflow array, [lo, sp) in LDS

  static __device__ __forceinline__ unsigned long long pack(uint32_t base, uint32_t mask) {
    return (static_cast<unsigned long long>(mask) << 32) | base;
  }
  __device__ __forceinline__ void push(uint32_t base, uint32_t mask) {
    if (sp >= kStackDepth) return;  // unreachable: the builders refuse trees that need more entries
    if (sp - lo == kLdsStack) {
      const unsigned long long e = ring[(lo & (kLdsStack - 1)) * kTraceBlock];
      ov[lo] = make_uint2(uint32_t(e), uint32_t(e >> 32));
      lo++;
    }
    ring[(sp & (kLdsStack - 1)) * kTraceBlock] = pack(base, mask);
    sp++;
  }
  __device__ __forceinline__ void pop(uint32_t& base, uint32_t& mask) {
    sp--;
    if (sp < lo) {
      lo = sp;
      const uint2 e = ov[sp];
      base = e.x;
      mask = e.y;
    } else {
      const unsigned long long e = ring[(sp & (kLdsStack - 1)) * kTraceBlock];
      base = uint32_t(e);
      mask = uint32_t(e >> 32);
    }
  }
};

// The closest hit is the minimum of (t, primitive) over the primitives that
// accept the ray's whole segment, whatever order they are tested in (when a
// wave tests them depends on its other rays): an unsigned key in that order (t
// may be negative where tmin is).  Only boxes are tested against the closest
// hit so far.  A triangle is not: it accepts by T <= |den| * tfar, and at t =
// T / |den| itself |den| * t may round below T, so one of two coincident
// triangles would be dropped or kept by the order of the tests.
__device__ __forceinline__ unsigned long long hit_key(float t, uint32_t prim) {
  const uint32_t u = __float_as_uint(t);
  return (static_cast<unsigned long long>(u ^ (uint32_t(int32_t(u) >> 31) | 0x80000000u)) << 32) | prim;
}
__device__ __forceinline__ float key_t(unsigned long long key) {
  const uint32_t u = uint32_t(key >> 32);
  return __uint_as_float(u ^ (uint32_t(~int32_t(u) >> 31) | 0x80000000u));
}

struct TraceRay {
  f3 o, d;
  f3 inv;          // 1 / d, components below 1e-18 in magnitude raised to it (sign kept)
  uint32_t oct;    // negative axes: bit 4 x, bit 5 y, bit 6 z (the address bits of a node's plane chunks)
  float tmin, tfar;  // tfar: the closest hit's distance once there is one
  uint32_t node;
  uint32_t gbase, gmask;  // current group: first inner child; bits 0-7 children to visit, in visiting order; 8-15 inner mask
  uint32_t hitp;   // primitive record of the closest hit, kNoHit: none
  Hit h;           // filled by trace_finish
  static constexpr uint32_t kNoHit = 0xffffffffu;
  __device__ __forceinline__ bool hit() const { return hitp != kNoHit; }
  // Without a hit any key is closer: t = T / |den| may round above the tmax
  // that T <= |den| * tmax was accepted with.
  __device__ __forceinline__ unsigned long long key() const { return hit() ? hit_key(tfar, hitp) : ~0ull; }
};

// Fills the hit record of a finished closest-hit traversal.
__device__ __forceinline__ void trace_finish(const DevScene& s, TraceRay& r) {
  if (r.hit()) {
    prim_hit(s, r.hitp, r.o, r.d, r.tfar, r.h);
  } else {
    r.h.t = r.tfar;
    r.h.u = r.h.v = 0.f;
    r.h.prim = 0;
    r.h.geom = 0xffffffffu;
  }
}

// A closest-hit traversal interrupted at a launch's visit budget: the node
// to visit next, the current group and the pending ones, the closest hit so
// far.  Resuming it replays nothing, so the result is the one an
// uninterrupted traversal gives.
struct ResumeState {
  uint32_t node, sp, gbase, gmask, hitp;
  float tfar;
  uint32_t pad[2];
  uint2 stack[kStackDepth];
};

__device__ inline void save_trace(ResumeState& rs, const TraceRay& r, const TraceStack& st) {
  rs.node = r.node;
  rs.sp = uint32_t(st.sp);
  rs.gbase = r.gbase;
  rs.gmask = r.gmask;
  rs.hitp = r.hitp;
  rs.tfar = r.tfar;
  for (int k = 0; k < st.sp; k++) {
    if (k < st.lo) {
      rs.stack[k] = st.ov[k];
    } else {
      const unsigned long long e = st.ring[(k & (kLdsStack - 1)) * kTraceBlock];
      rs.stack[k] = make_uint2(uint32_t(e), uint32_t(e >> 32));
    }
  }
}

// After trace_begin on the same ray.
__device__ inline void restore_trace(const ResumeState& rs, TraceRay& r, TraceStack& st) {
  r.node = rs.node;
  r.gbase = rs.gbase;
  r.gmask = rs.gmask;
  r.hitp = rs.hitp;
  r.tfar = rs.tfar;
  const int n = min(int(rs.sp), kStackDepth);
  for (int k = 0; k < n; k++) st.push(rs.stack[k].x, rs.stack[k].y);
}

__device__ __forceinline__ void trace_begin(TraceRay& r, TraceStack& st, f3 o, f3 d, float tmin, float tmax) {
  r.o = o;
  r.d = d;
  // A zero direction component would make the slab arithmetic produce
  // inf - inf; a tiny one of the same sign keeps every slab finite.
  const auto safe = [](float x) { return fabsf(x) < 1e-18f ? copysignf(1e-18f, x) : x; };
  r.inv = mk(1.0f / safe(d.x), 1.0f / safe(d.y), 1.0f / safe(d.z));
  r.oct = (r.inv.x < 0.f ? 16u : 0u) | (r.inv.y < 0.f ? 32u : 0u) | (r.inv.z < 0.f ? 64u : 0u);
  r.tmin = tmin;
  r.tfar = tmax;
  r.node = 0;
  r.gbase = r.gmask = 0;
  r.hitp = TraceRay::kNoHit;
  st.sp = 0;
  st.lo = 0;
}

// Orders the wave's LDS accesses around the pooled tests: LDS executes one
// wave's instructions in order, so only the compiler needs holding back.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Leaf children of one node hit by a ray: their mask (slots) and where their
// primitives are.
struct LeafGroup {
  uint32_t prim_base, ends0, ends1, hits;
};

// Bits [begin, end) of the node's primitives for every hit leaf slot.
__device__ __forceinline__ uint32_t leaf_prims(const LeafGroup& g) {
  const unsigned long long ends = (static_cast<unsigned long long>(g.ends1) << 32) | g.ends0;
  const unsigned long long begins = ends << 8;
  uint32_t pm = 0;
  for (uint32_t h = g.hits; h; h &= h - 1u) {
    const uint32_t sh = 8u * uint32_t(__ffs(int(h)) - 1);
    const uint32_t b = uint32_t(begins >> sh) & 0xffu, c = (uint32_t(ends >> sh) & 0xffu) - b;
    if (c) pm |= (0xffffffffu >> (32u - c)) << b;
  }
  return pm;
}

// Visit node r.node: test its eight child boxes, make the hit inner children
// the current group and choose the node to visit next.  leaf: the hit leaf
// children, for the caller to intersect.  Returns false when no node is left.
//
// Bound by instruction issue (the loads hide behind the other waves): a child
// costs six v_fma_mix_f32 straight from the packed planes, two three-way and
// two two-way min / max, one fused multiply-add of slack and one compare.
//
// FAR: byte offsets of nodes need 64 bits (a tree of 4 GiB or more).  Without
// it a chunk's address is a scalar base and one 32-bit register.
template <bool FAR>
__device__ __forceinline__ bool trace_node(const DevScene& s, TraceRay& r, TraceStack& st, LeafGroup& leaf) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  const uint32_t sx = r.oct & 16u, sy = r.oct & 32u, sz = r.oct & 64u;
  uint4 hdr, nx, fx, ny, fy, nz, fz, hb;
  const auto load = [&](const char* nodes, auto off) {  // the chunks' bits are clear in off: | is +
    const auto at = [&](auto k, int fixed) { return *reinterpret_cast<const uint4*>(nodes + k + fixed); };
    hdr = at(off, 0x20);
    nx = at(off | sx, 0), fx = at(off | (sx ^ 16u), 0);
    ny = at(off | sy, 0x40), fy = at(off | (sy ^ 32u), 0x40);
    nz = at(off | sz, 0x30), fz = at(off | (sz ^ 64u), 0x30);
    hb = at(off, 0x50);
  };
  if constexpr (FAR)
    load(reinterpret_cast<const char*>(s.wnodes), size_t(r.node) << 7);
  else
    load(reinterpret_cast<const char*>(s.wnodes), r.node << 7);
  // A child plane at offset q along x lies at origin + q * step; its ray
  // parameter is q * (step / d) + (origin - o) / d, the step a power of two,
  // so the first factor is exact.
  const float ax = quant_step(hdr.w) * r.inv.x, ay = quant_step(hdr.w >> 8) * r.inv.y,
              az = quant_step(hdr.w >> 16) * r.inv.z;
  const float bx = (__uint_as_float(hdr.x) - r.o.x) * r.inv.x, by = (__uint_as_float(hdr.y) - r.o.y) * r.inv.y,
              bz = (__uint_as_float(hdr.z) - r.o.z) * r.inv.z;
  uint32_t hits = 0;
  const uint32_t wnx[4] = {nx.x, nx.y, nx.z, nx.w}, wny[4] = {ny.x, ny.y, ny.z, ny.w}, wnz[4] = {nz.x, nz.y, nz.z, nz.w};
  const uint32_t wfx[4] = {fx.x, fx.y, fx.z, fx.w}, wfy[4] = {fy.x, fy.y, fy.z, fy.w}, wfz[4] = {fz.x, fz.y, fz.z, fz.w};
#pragma unroll
  for (int w = 0; w < 4; w++) {
    const h2 hnx = __builtin_bit_cast(h2, wnx[w]), hny = __builtin_bit_cast(h2, wny[w]), hnz = __builtin_bit_cast(h2, wnz[w]);
    const h2 hfx = __builtin_bit_cast(h2, wfx[w]), hfy = __builtin_bit_cast(h2, wfy[w]), hfz = __builtin_bit_cast(h2, wfz[w]);
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const float tnx = fmaf(float(hnx[c]), ax, bx), tfx = fmaf(float(hfx[c]), ax, bx);
      const float tny = fmaf(float(hny[c]), ay, by), tfy = fmaf(float(hfy[c]), ay, by);
      const float tnz = fmaf(float(hnz[c]), az, bz), tfz = fmaf(float(hfz[c]), az, bz);
      const float tn = fmaxf(fmaxf(fmaxf(tnx, tny), tnz), r.tmin);
      float tf = fminf(fminf(fminf(tfx, tfy), tfz), r.tfar);
      tf = fmaf(fabsf(tf), 9.6e-7f, tf);  // slack for the rounding of the slab arithmetic on both sides
      hits |= tn <= tf ? 1u << (2 * w + c) : 0u;
    }
  }
  const uint32_t imask = hdr.w >> 24;
  leaf.hits = hits & ~imask;
  leaf.prim_base = hb.y;
  leaf.ends0 = hb.z;
  leaf.ends1 = hb.w;
  const uint32_t o = r.oct >> 4;
  uint32_t g = hits & imask;
  if (g) {
    if (r.gmask & 0xffu) st.push(r.gbase, r.gmask);
    // bit slot -> bit slot ^ o, so the lowest set bit is the child to visit first
    g = ((g & 0xaau) >> (o & 1u)) | ((g & 0x55u) << (o & 1u));
    g = ((g & 0xccu) >> (o & 2u)) | ((g & 0x33u) << (o & 2u));
    g = ((g & 0xf0u) >> (o & 4u)) | ((g & 0x0fu) << (o & 4u));
    r.gbase = hb.x;
    r.gmask = g | imask << 8;
  } else if (!(r.gmask & 0xffu)) {
    if (st.sp == 0) return false;
    st.pop(r.gbase, r.gmask);
  }
  const uint32_t slot = uint32_t(__ffs(int(r.gmask)) - 1) ^ o;
  r.gmask &= r.gmask - 1u;
  r.node = r.gbase + uint32_t(__popc(r.gmask & (((1u << slot) - 1u) << 8)));
  return true;
}

// Sum of v over the lanes below this one (all 64 lanes active).
__device__ __forceinline__ uint32_t wave_exclusive_sum(uint32_t v) {
  int x = int(v);
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return uint32_t(x) - v;
}

// Items of a launch for the lanes of a wave, consecutive ones together.  A
// wave's first share is its own by position and only the rest is dealt out in
// chunks, one atomic each: a counter takes about 11 ns per atomic (and a load
// of it waits as long) whoever asks, so with one per wave and 64 items an
// extension launch of a million rays over a small tree took 263 us, now 150,
// and an empty launch of 8192 waves 95 us.  A block asks a used-up counter once.
// All members are wave-uniform.
struct ItemDealer {
  uint32_t n, base, left;   // items in all; the wave's own
  uint32_t dealt, chunk;    // items given out by position; of one later chunk
  uint32_t* ctr;            // later chunks (nullptr: none)
  lds_u32* used_up;         // set once the counter has no more for this block
  bool exhausted;           // nothing left beyond the wave's own

  // wave: this wave's number; those from `waves` on get nothing
  __device__ __forceinline__ void start(uint32_t items, uint32_t* counter, lds_u32* flag, uint32_t wave, uint32_t waves,
                                        uint32_t share, uint32_t later) {
    n = items;
    ctr = counter;
    used_up = flag;
    chunk = later;
    const unsigned long long b = static_cast<unsigned long long>(wave) * share;
    base = uint32_t(b);
    left = wave < waves && b < n ? min(share, uint32_t(n - b)) : 0u;
    dealt = uint32_t(min(static_cast<unsigned long long>(waves) * share, static_cast<unsigned long long>(n)));
    exhausted = !ctr || wave >= waves || dealt == n;
  }
  __device__ __forceinline__ bool more() const { return !exhausted || left > 0; }
  // The next item for each lane of `need`; n or more: none.
  __device__ __forceinline__ uint32_t take(unsigned long long need, uint32_t lane) {
    const uint32_t want = (uint32_t)__popcll(need);
    const uint32_t rank = (uint32_t)__popcll(need & ((1ull << lane) - 1ull));
    uint32_t nbase = 0, nleft = 0;
    if (left < want && !exhausted) {
      uint32_t b = n;
      if (!*(volatile lds_u32*)used_up) {
        if (lane == 0) b = atomicAdd(ctr, chunk);
        b = __builtin_amdgcn_readfirstlane(b) + dealt;  // scalar, as are the loops that depend on it
        if (b >= n) *(volatile lds_u32*)used_up = 1u;
      }
      b = __builtin_amdgcn_readfirstlane(b);
      if (b >= n) {
        exhausted = true;
      } else {
        nbase = b;
        nleft = min(chunk, n - b);
        if (n - b <= chunk) exhausted = true;
      }
    }
    uint32_t i = 0xffffffffu;
    if (rank < left)
      i = base + rank;
    else if (rank - left < nleft)
      i = nbase + (rank - left);
    const uint32_t fromOld = min(want, left);
    base += fromOld;
    left -= fromOld;
    if (nleft) {
      const uint32_t fromNew = min(want - fromOld, nleft);
      base = nbase + fromNew;
      left = nleft - fromNew;
    }
    return i;
  }
};
// Shares of a launch of n items over `waves` resident waves: two fifths by
// position, the rest in chunks of a third of the mean.  All by position left a
// frame's first launch waiting for the waves that own its costliest part (1080p
// large mesh, extension rays 57.9 -> 86 ms), chunks of an eighth and less
// waited on the counter (volume 15.0 -> 21.0 ms).
__device__ __forceinline__ void deal_shares(uint32_t n, uint32_t waves, uint32_t& share, uint32_t& chunk) {
  const uint32_t mean = (n + waves - 1) / waves;
  share = max(64u, (mean * 2u / 5u + 63u) & ~63u);
  chunk = min(max(mean / 3u, 64u), 512u);
}

// Stream traversal for kernels that own a batch of rays.  Rays end at
// different steps, so a lane that has none takes the next of the batch while
// the others continue; and about one lane-step in nine reaches leaves, so a
// wave queues the leaf groups its lanes find and intersects their primitives
// together, 64 at a time, once enough have gathered (flush_leaves).
//
// Rays: dealt out by ItemDealer, from the counter `fetch`; with fetch ==
// nullptr, wave w of the grid owns the items [w * per_wave, (w + 1) * per_wave).
// Job: bool load(uint32_t i, f3& o, f3& d, float& tmin, float& tmax, uint32_t& tag)
//      void finish(uint32_t i, uint32_t tag, const TraceRay& r)
//      static constexpr bool kTagIsIndex; with it the tag is the item index
//      i itself, and the stream keeps one register for both
//      static constexpr bool kSuspend; with it, a ray that has visited
//      job.budget nodes in this launch is offered to the job, which may keep
//      it for a later launch (per-ray costs are heavy-tailed: near-grazing
//      rays over dense meshes visit thousands of nodes, and a launch cannot
//      end before its slowest ray):
//      uint32_t budget;
//      void resume(uint32_t tag, TraceRay& r, TraceStack& st)   (after trace_begin)
//      bool suspend(uint32_t tag, const TraceRay& r, const TraceStack& st)
// Launch with kTraceBlock threads per block; every lane must call this.
constexpr uint32_t kGroupFlush = 24;                // queued leaf groups at which a wave tests them
constexpr uint32_t kGroupQueue = kGroupFlush + 64;  // a step adds at most one group per lane
constexpr uint32_t kPoolSize = kTracePool;
// Waves that a launch's rays are spread over before a wave fills all its lanes
// (two per SIMD: 1024 to 4096 measured alike, without it a 64x48 render's
// traversal took 8 % longer) and fewest lanes of a wave.
constexpr uint32_t kSpreadWaves = 2048, kMinLanes = 8;
// Waves that rays are dealt to: those resident at once where the kernel has the
// device to itself, five per SIMD (the traversal kernels' registers) on 256 CUs.
// A grid of more (trace_blocks_per_cu above 5) only adds waves that start
// and leave.
constexpr uint32_t kResidentWaves = 5 * 4 * 256;

template <bool ANY, bool FAR, class Job>
__device__ __forceinline__ void trace_stream(const DevScene& s, uint32_t n, uint32_t* fetch, uint32_t per_wave, Job& job) {
  __shared__ unsigned long long lds_ring[kLdsStack * kTraceBlock];
  __shared__ u32x4 lds_group[kTraceBlock / 64][kGroupQueue];
  __shared__ u32x2 lds_pool[kTraceBlock / 64][kPoolSize];
  __shared__ unsigned long long lds_key[kTraceBlock];
  __shared__ float lds_tmax[kTraceBlock];  // end of each lane's segment
  __shared__ uint32_t lds_used_up;  // the counter has no more items for this block
  const uint32_t lane = __lane_id();
  const unsigned long long below = (1ull << lane) - 1ull;
  const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  lds_u4* const group = (lds_u4*)lds_group[wv];
  lds_u2* const pool = (lds_u2*)lds_pool[wv];
  lds_u64* const key = (lds_u64*)&lds_key[wv * 64];
  lds_f32* const seg = (lds_f32*)&lds_tmax[wv * 64];
  TraceOverflow ov;
  TraceStack st;
  st.ring = (lds_u64*)(lds_ring + threadIdx.x);
  st.ov = ov.e;
  TraceRay r;
  // A lane's ray is being traversed (active), waits for queued leaf groups of
  // its own with no node left (pend only), or has ended (have only).
  bool have = false, active = false, pend = false;
  uint32_t idx = 0, tag = 0, visits = 0;
  uint32_t queued = 0;            // leaf groups queued by the wave (wave-uniform)
  // With few rays a wave fills only some of its lanes, so that they spread over
  // the chip: a wave's step takes the longer the more lanes it has (more of
  // them reach leaves), and a launch cannot end before its slowest wave.
  const uint32_t wave = blockIdx.x * (kTraceBlock / 64) + wv;
  uint32_t lanes, share, chunk = 0, waves = gridDim.x * (kTraceBlock / 64);
  if (!fetch) {
    share = per_wave;
    lanes = min(64u, per_wave);
  } else {
    waves = min(waves, kResidentWaves);
    lanes = min(64u, max(kMinLanes, (n + kSpreadWaves - 1) / kSpreadWaves));
    deal_shares(n, waves, share, chunk);
    if (lanes < 64) share = chunk = lanes;
  }
  if (threadIdx.x == 0) lds_used_up = 0u;
  __syncthreads();
  ItemDealer items;
  items.start(n, fetch, (lds_u32*)&lds_used_up, wave, waves, share, chunk);
  const unsigned long long usable = ~0ull >> (64 - lanes);
  const uint32_t refill = lanes * 3 / 4;                    // refill once fewer lanes than this have a ray in flight
  const uint32_t flush = min(kGroupFlush, lanes * 3 / 8);  // queued leaf groups at which the wave tests them
  for (;;) {
    // Finished closest-hit rays are written out here, together: a wave's 64
    // rays end a few at a time, and recomputing and storing the hit in the
    // step in which its ray ended ran that code with about four lanes active
    // in nearly every step (1080p large-mesh frame, on
    // 4-wide nodes, 145.6 -> 138.0 ms).  An
    // any-hit ray has one byte or nothing to write and does so when it ends.
    if (!ANY && have && !active && !pend) {
      trace_finish(s, r);
      job.finish(Job::kTagIsIndex ? tag : idx, tag, r);
      have = false;
    }
    if (items.more()) {
      const unsigned long long need = __ballot(!have) & usable;
      if (need) {
        const uint32_t i = items.take(need, lane);
        if ((need >> lane & 1ull) && i < n) {
          f3 o, d;
          float tmin, tmax;
          if (job.load(i, o, d, tmin, tmax, tag)) {
            if constexpr (!Job::kTagIsIndex) idx = i;
            trace_begin(r, st, o, d, tmin, tmax);
            seg[lane] = tmax;
            if constexpr (Job::kSuspend) job.resume(tag, r, st);
            visits = 0;
            have = active = true;
          }
        }
      }
    }
    if (__ballot(have) == 0ull) {
      if (!items.more()) break;  // every finished ray was written out above
      continue;
    }
    for (;;) {
      LeafGroup leaf;
      leaf.hits = 0;
      if (active) active = trace_node<FAR>(s, r, st, leaf);
      const unsigned long long found = __ballot(leaf.hits != 0);
      if (found) {
        if (leaf.hits) {
          const uint32_t k = queued + (uint32_t)__popcll(found & below);
          group[k] = u32x4{leaf.prim_base, leaf.ends0, leaf.ends1, leaf.hits | lane << 8};
          pend = true;
        }
        queued += (uint32_t)__popcll(found);
      }
      if constexpr (Job::kSuspend) {
        if (active && ++visits >= job.budget && !pend) {
          if (job.suspend(tag, r, st)) have = active = false;
          visits = 0;
        }
      }
      uint32_t busy = (uint32_t)__popcll(__ballot(active));
      const uint32_t waiting = (uint32_t)__popcll(__ballot(pend && !active));
      // Test the queued primitives when a wave's worth has gathered, or when
      // the lanes that can do nothing else outnumber a third of the others.
      if (queued >= flush || 3 * waiting > busy) {
        key[lane] = ~0ull;
        wave_lds_fence();
        for (uint32_t g0 = 0; g0 < queued; g0 += 64) {
          uint32_t pm = 0, base = 0, owner = 0;
          if (g0 + lane < queued) {
            const u32x4 e = group[g0 + lane];
            const LeafGroup lg{e.x, e.y, e.z, e.w & 0xffu};
            pm = leaf_prims(lg);
            base = e.x;
            owner = e.w >> 8;
          }
          while (__ballot(pm != 0)) {
            const uint32_t t = (uint32_t)__popc(pm);
            const uint32_t pre = wave_exclusive_sum(t);
            const uint32_t total = __builtin_amdgcn_readlane(pre + t, 63);
            const uint32_t cap = s.pool_cap;
            const uint32_t fit = min(t, cap - min(pre, cap));  // entries beyond the pool wait for the next round
            for (uint32_t k = 0; k < fit; k++) {
              pool[pre + k] = u32x2{base + uint32_t(__ffs(int(pm)) - 1), owner};
              pm &= pm - 1u;
            }
            wave_lds_fence();
            const bool valid = lane < min(total, cap);
            u32x2 e = {0u, lane};
            if (valid) e = pool[lane];
            // the owner's ray, read from its registers
            const f3 o = mk(__shfl(r.o.x, e.y), __shfl(r.o.y, e.y), __shfl(r.o.z, e.y));
            const f3 d = mk(__shfl(r.d.x, e.y), __shfl(r.d.y, e.y), __shfl(r.d.z, e.y));
            const float tmin = __shfl(r.tmin, e.y);
            float th = seg[e.y];
            if (valid && isect_prim(s, e.x, o, d, tmin, th)) {
              if (ANY)
                key[e.y] = 0;
              else
                __hip_atomic_fetch_min(&key[e.y], hit_key(th, e.x), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
            }
            wave_lds_fence();
          }
        }
        queued = 0;
        pend = false;
        const unsigned long long k = key[lane];
        if (ANY) {
          if (have && k == 0) {
            r.hitp = 0;
            active = false;
          }
        } else if (have && k < r.key()) {
          r.tfar = key_t(k);
          r.hitp = uint32_t(k);
        }
        wave_lds_fence();
        busy = (uint32_t)__popcll(__ballot(active));
      }
      if (ANY && have && !active && !pend) {
        job.finish(Job::kTagIsIndex ? tag : idx, tag, r);
        have = false;
      }
      if (busy == 0 && queued == 0) break;
      if (items.more() && (uint32_t)__popcll(__ballot(active || pend)) < refill) break;
    }
  }
}

// Single-ray traversal for kernels that trace a data-dependent number of rays
// per lane (launched with at most kTraceBlock threads per block).
template <bool ANY>
__device__ __forceinline__ bool trace(const DevScene& s, f3 o, f3 d, float tmin, float tmax, Hit& h) {
  __shared__ unsigned long long lds_ring1[kLdsStack * kTraceBlock];

  TraceRay r;
  TraceOverflow ov;
  TraceStack st;
  st.ring = (lds_u64*)(lds_ring1 + threadIdx.x);
  st.ov = ov.e;
  trace_begin(r, st, o, d, tmin, tmax);
  // lanes loop independently here, so each tests its own primitives
  for (bool more = true; more;) {
    LeafGroup leaf;
    more = trace_node<true>(s, r, st, leaf);
    if (leaf.hits) {
      for (uint32_t pm = leaf_prims(leaf); pm; pm &= pm - 1u) {
        const uint32_t p = leaf.prim_base + uint32_t(__ffs(int(pm)) - 1);
        float t = tmax;
        if (!isect_prim(s, p, r.o, r.d, r.tmin, t)) continue;
        if (hit_key(t, p) < r.key()) {
          r.tfar = t;
          r.hitp = p;
        }
        if (ANY) {
          more = false;
          break;
        }
      }
    }
  }
  if (!ANY) trace_finish(s, r);
  h = r.h;
  return r.hit();
}

}  // namespace rad
