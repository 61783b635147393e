// Traversal kernels: the extension and shadow rays of the wavefront
// integrators and the ray-batch entry points (accel/embree.cpp:79-111).
#include <algorithm>

#include "wavefront.h"

namespace rad {

// The tag of an extend ray is its queue position; its state index is base + tag.
struct ExtendJob {
  static constexpr bool kSuspend = true;
  static constexpr bool kTagIsIndex = true;
  uint32_t base;
  const float4* ray;
  float4* hit;
  uint32_t* hit_geom;
  uint32_t* susp;                 // null: traversals run to the end
  const ResumeState* rin;         // pool this launch resumes from
  ResumeState* rout;              // pool this launch suspends into
  uint32_t* rcount;               // entries of rout
  uint32_t cap, budget;
  __device__ __forceinline__ void resume(uint32_t i, TraceRay& r, TraceStack& st) {
    if (!susp) return;
    const uint32_t s = base + i;
    const uint32_t j = susp[s];
    if (j == kNoSusp) return;
    restore_trace(rin[j], r, st);
    susp[s] = kNoSusp;
  }
  __device__ __forceinline__ bool suspend(uint32_t i, const TraceRay& r, const TraceStack& st) {
    const uint32_t j = atomicAdd(rcount, 1u);
    if (j >= cap) return false;  // pool full: the ray finishes in this launch
    save_trace(rout[j], r, st);
    susp[base + i] = j;
    return true;
  }
  __device__ __forceinline__ bool load(uint32_t i, f3& o, f3& d, float& tmin, float& tmax, uint32_t& tag) {
    float4 a = ray[2 * size_t(i)], b = ray[2 * size_t(i) + 1];
    o = mk(a.x, a.y, a.z);
    d = mk(b.x, b.y, b.z);
    tmin = a.w;
    tmax = b.w;
    tag = i;
    return true;
  }
  // hits are stored by extend-queue position: consecutive rays of the
  // queue write consecutive entries, and classify reads them in order
  __device__ __forceinline__ void finish(uint32_t i, uint32_t, const TraceRay& r) {
    hit[i] = make_float4(r.h.t, r.h.u, r.h.v, __uint_as_float(r.hit() ? r.h.prim : 0u));
    hit_geom[i] = r.hit() ? r.h.geom : 0xffffffffu;
  }
};

// The traversal kernels are capped at 96 VGPRs (five waves per SIMD; nothing
// spills, two to five registers with 64-bit node addresses): they wait on node
// loads more than half of a wave's time, and resident waves hide that.  1080p 64-spp large-mesh frame, extension rays
// 62.8 ms at four waves, 62.5 at five, 74.3 at six (42 registers spill).  Over
// the 4-wide tree with primitives tested every step they took 68 ms
// (0.88 of the SIMD cycles issuing, 0.46 of the lanes active; now 0.62 and
// 0.65); 3 M incoherent rays 776 -> 353 us, 4 M occlusion rays 755 -> 369 us.
template <bool FAR>
__global__ void __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(5))) k_extend(Wavefront w, DevScene scene, int in) {
  ExtendJob job{state_index(w.Q, in, 0), w.ray[in], w.hit, w.hit_geom, w.susp, w.resume[in], w.resume[1 - in],
                &w.cnt[CNT_SUSP + 1 - in], w.resume_cap, w.susp ? w.visit_budget : 0xffffffffu};
  trace_stream<false, FAR>(scene, w.cnt[in], &w.cnt[CNT_FETCH_EXT], 0, job);
}

struct ShadowJob {
  static constexpr bool kSuspend = false;
  static constexpr bool kTagIsIndex = false;
  const float4 *sh_o, *sh_d, *sh_c;
  SlotField<float4> lsum;
  __device__ __forceinline__ bool load(uint32_t i, f3& o, f3& d, float& tmin, float& tmax, uint32_t& tag) {
    float4 a = sh_o[i], b = sh_d[i];
    o = mk(a.x, a.y, a.z);
    d = mk(b.x, b.y, b.z);
    tmin = 0.f;
    tmax = a.w;
    tag = __float_as_uint(b.w);
    return true;
  }
  __device__ __forceinline__ void finish(uint32_t i, uint32_t s, const TraceRay& r) {
    if (r.hit()) return;  // occluded
    float4 c = sh_c[i];
    float4 l = lsum[s];
    lsum[s] = make_float4(l.x + c.x, l.y + c.y, l.z + c.z, l.w);
  }
};

template <bool FAR>
__global__ void __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(5))) k_shadow(Wavefront w, DevScene scene) {
  ShadowJob job{w.sh_o, w.sh_d, w.sh_c, w.lsum};
  trace_stream<true, FAR>(scene, w.cnt[CNT_SHADOW], &w.cnt[CNT_FETCH_SH], 0, job);
}

struct ClosestJob {
  static constexpr bool kSuspend = false;
  static constexpr bool kTagIsIndex = false;
  const float4* rays;
  float* hits;
  __device__ __forceinline__ bool load(uint32_t i, f3& o, f3& d, float& tmin, float& tmax, uint32_t& tag) {
    float4 a = rays[2 * i], b = rays[2 * i + 1];
    o = mk(a.x, a.y, a.z);
    d = mk(b.x, b.y, b.z);
    tmin = a.w;
    tmax = b.w;
    tag = __float_as_uint(b.w);
    return true;
  }
  __device__ __forceinline__ void finish(uint32_t i, uint32_t tmax_bits, const TraceRay& r) {
    float* o = hits + 5 * size_t(i);
    o[0] = r.hit() ? r.h.t : __uint_as_float(tmax_bits);
    o[1] = r.hit() ? r.h.u : 0.f;
    o[2] = r.hit() ? r.h.v : 0.f;
    o[3] = __uint_as_float(r.hit() ? r.h.prim : 0xffffffffu);
    o[4] = __uint_as_float(r.hit() ? r.h.geom : 0xffffffffu);
  }
};

struct AnyJob {
  static constexpr bool kSuspend = false;
  static constexpr bool kTagIsIndex = false;
  const float4* rays;
  uint8_t* occ;
  __device__ __forceinline__ bool load(uint32_t i, f3& o, f3& d, float& tmin, float& tmax, uint32_t& tag) {
    float4 a = rays[2 * i], b = rays[2 * i + 1];
    o = mk(a.x, a.y, a.z);
    d = mk(b.x, b.y, b.z);
    tmin = a.w;
    tmax = b.w;
    tag = 0;
    return true;
  }
  __device__ __forceinline__ void finish(uint32_t i, uint32_t, const TraceRay& r) { occ[i] = r.hit() ? 1 : 0; }
};

template <bool FAR>
__global__ void __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(5))) k_closest(DevScene scene, const float4* rays, uint32_t n, uint32_t per_wave,
                                                          float* hits) {
  ClosestJob job{rays, hits};
  trace_stream<false, FAR>(scene, n, nullptr, per_wave, job);
}

template <bool FAR>
__global__ void __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(5))) k_any(DevScene scene, const float4* rays, uint32_t n, uint32_t per_wave,
                                                      uint8_t* occ) {
  AnyJob job{rays, occ};
  trace_stream<true, FAR>(scene, n, nullptr, per_wave, job);
}

void LaunchExtend(const Wavefront& w, const DevScene& scene, int in, const LaunchCfg& c, hipStream_t s) {
  hipLaunchKernelGGL(scene.wide_far ? k_extend<true> : k_extend<false>, dim3(c.trace_blocks), dim3(kTraceBlock), 0, s, w, scene, in);
}
void LaunchShadow(const Wavefront& w, const DevScene& scene, const LaunchCfg& c, hipStream_t s) {
  hipLaunchKernelGGL(scene.wide_far ? k_shadow<true> : k_shadow<false>, dim3(c.trace_blocks), dim3(kTraceBlock), 0, s, w, scene);
}
// Rays a wave of a ray batch owns.  A wave drains at the end of its share with
// few lanes busy, so the shares are as large as still gives about four waves
// per SIMD (3 M closest-hit rays: 64 per wave 601 us, 256 402, 1024 366, 4096
// waves 353), and small batches spread over the chip in part-filled waves.
static uint32_t PerWave(uint32_t n) { return std::max(16u, (n + 4095u) / 4096u); }
static unsigned BatchBlocks(uint32_t n, uint32_t per) {
  return unsigned((n + uint64_t(per) * (kTraceBlock / 64) - 1) / (uint64_t(per) * (kTraceBlock / 64)));
}
void LaunchClosest(const DevScene& scene, const void* rays, uint32_t n, void* hits, hipStream_t s) {
  const uint32_t per = PerWave(n);
  if (n)
    hipLaunchKernelGGL(scene.wide_far ? k_closest<true> : k_closest<false>, dim3(BatchBlocks(n, per)), dim3(kTraceBlock), 0, s,
                       scene, (const float4*)rays, n, per, (float*)hits);
}
void LaunchAny(const DevScene& scene, const void* rays, uint32_t n, uint8_t* occ, hipStream_t s) {
  const uint32_t per = PerWave(n);
  if (n)
    hipLaunchKernelGGL(scene.wide_far ? k_any<true> : k_any<false>, dim3(BatchBlocks(n, per)), dim3(kTraceBlock), 0, s, scene,
                       (const float4*)rays, n, per, occ);
}

}  // namespace rad
