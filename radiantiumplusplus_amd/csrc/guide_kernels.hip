// FP16 MFMA kernels of the guiding network: inference for probe inputs, one
// training step (forward, loss, backward, weight gradients), and the Adam
// update of the FP32 master weights.  (Inference for path vertices is in
// the path kernels; both use the forward pass of guide_mlp.h.)
#include <algorithm>
#include <cmath>
#include <random>
#include <stdexcept>
#include <vector>

#include "guide_dev.h"
#include "guide_mlp.h"
#include "guide_state.h"
#include "scene_host.h"

namespace rad {
namespace guide {

// Inference over n vertices: feats (9 floats per vertex) -> raw outputs
// (48 halves) at raw[slot_of[i] * 48] (or raw[i * 48] without slot_of).
__global__ void __launch_bounds__(256) k_guide_infer(GuideNet net, const float* feats, const uint32_t* n_dev, uint32_t n_host,
                                                     const uint32_t* slot_of, _Float16* raw) {
  __shared__ __align__(16) _Float16 sW[kWeights];
  __shared__ __align__(16) _Float16 sB[kBiases];
  load_weights_lds_frag(sW, sB, net.w, net.b);
  __syncthreads();
  const uint32_t n = n_dev ? *n_dev : n_host;
  const int lane = __lane_id();
  const int v = lane & 15, g = lane >> 4;
  const uint32_t wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  for (uint32_t tile = blockIdx.x * waves + wave; tile * 16 < n; tile += gridDim.x * waves) {
    uint32_t i = tile * 16 + v;
    float f9[kFeat];
    if (i < n) {
      for (int k = 0; k < kFeat; k++) f9[k] = feats[size_t(i) * kFeat + k];
    } else {
      for (int k = 0; k < kFeat; k++) f9[k] = 0.f;
    }
    FeatScalars fs = feat_scalars(f9, net.lo, net.inv_ext);
    h4 out[3];
    infer_tile(sW, sB, fs, out);
    if (i < n) {
      size_t base = size_t(slot_of ? slot_of[i] : i) * kOut;
#pragma unroll
      for (int t = 0; t < 3; t++) *reinterpret_cast<h4*>(raw + base + 16 * t + 4 * g) = out[t];
    }
  }
}

// Per-record loss gradient with respect to the 40 raw outputs, for
// loss_j = wn_j * (-log q(dir_j)), wn_j = min(w_j * wnorm, wmax).  The output
// gradients are kept in FP16 multiplied by kDzScale (undone in the weight
// gradient), so large sample weights stay inside the FP16 range.
constexpr float kDzScale = 1.f / 32.f;

// Reductions over the four lanes of a record (v, v + 16, v + 32, v + 48).
__device__ __forceinline__ float record_max(float x) {
  x = fmaxf(x, __shfl_xor(x, 16));
  return fmaxf(x, __shfl_xor(x, 32));
}
__device__ __forceinline__ float record_sum(float x) {
  x += __shfl_xor(x, 16);
  return x + __shfl_xor(x, 32);
}

// Lobe l points from the vertex p to the target c + h * (raw means).  Lane
// group g of a record's four has the lobes 2 g and 2 g + 1 (raw and d: their
// outputs); the loss is the same in all four.
__device__ __forceinline__ float record_loss_grad(const float* raw, f3 dir, float wn, f3 p, f3 cen, f3 half,
                                                  float d[2 * kRawPerLobe]) {
  constexpr int N = kLobes / 4;
  float a[N], logv[N], kap[N], c[N], len[N], lp[N];
  f3 mu[N];
  bool kin[N];
  float mx = -kInf;
#pragma unroll
  for (int l = 0; l < N; l++) mx = fmaxf(mx, raw[kRawPerLobe * l]);
  mx = record_max(mx);
  float se = 0.f;
#pragma unroll
  for (int l = 0; l < N; l++) {
    a[l] = expf(raw[kRawPerLobe * l] - mx);
    se += a[l];
  }
  se = record_sum(se);
  float lm = -kInf;
#pragma unroll
  for (int l = 0; l < N; l++) {
    a[l] /= se;  // pi_l
    f3 m = lobe_vector(raw + kRawPerLobe * l, p, cen, half);
    len[l] = sqrtf(sqnorm(m));
    mu[l] = len[l] > 1e-6f ? m / len[l] : mk(0.f, 1.f, 0.f);
    float kr = raw[kRawPerLobe * l + 4];
    kin[l] = kr > -3.f && kr < 6.f;
    kap[l] = expf(fminf(fmaxf(kr, -3.f), 6.f));
    c[l] = dot(mu[l], dir);
    logv[l] = logf(kap[l]) - logf(2.f * kPi) - log1pf(-expf(-2.f * kap[l])) + kap[l] * (c[l] - 1.f);
    lp[l] = logf(a[l]) + logv[l];
    lm = fmaxf(lm, lp[l]);
  }
  lm = record_max(lm);
  float s = 0.f;
#pragma unroll
  for (int l = 0; l < N; l++) s += expf(lp[l] - lm);
  float logq = lm + logf(record_sum(s));
#pragma unroll
  for (int l = 0; l < N; l++) {
    float r = expf(lp[l] - logq);
    float k = kap[l];
    d[kRawPerLobe * l] = -wn * (r - a[l]);
    float e = expf(-2.f * k);
    float dlogv_dk = 1.f / k - 2.f * e / (1.f - e) + (c[l] - 1.f);
    d[kRawPerLobe * l + 4] = kin[l] ? -wn * r * dlogv_dk * k : 0.f;
    // d(log vMF) / d(target output) = (dir - mu c) kappa / |v| times h
    f3 gm = len[l] > 1e-6f ? mul(dir - mu[l] * c[l], half) * (k / len[l]) : splat(0.f);
    d[kRawPerLobe * l + 1] = -wn * r * gm.x;
    d[kRawPerLobe * l + 2] = -wn * r * gm.y;
    d[kRawPerLobe * l + 3] = -wn * r * gm.z;
  }
  return -wn * logq;
}

// Gradients of tiles of 64 records (4 waves x 16), summed over the records but
// not yet divided by the batch size: row blockIdx.x of `partial` (kTrainRow
// floats: the parameters, then the loss), which k_guide_train_sum adds up.
//
// The matrix products (4 GFLOP at 32768 records) are 5 us of the matrix cores; the
// kernel is bound by the chain of its phases (LDS operands, the loss, barriers)
// with one wave per SIMD, as the weights (both operand orders) and the
// activations of a tile fill the LDS.  So every matrix operand is stored in
// the order in which the lanes read it, one conflict-free 8-byte read each;
// the four lanes of a record share its lobes; and the gradient of a block's
// tiles stays in registers (100 per lane) and is written once: 512 blocks that
// added their tile's 20.6 K values to one gradient atomically, after operand
// reads from rows of 128 bytes (8 lanes to a bank), took 115 us at 32768
// records and 57.8 us at the 8192 of a training step; now 37 and 24.7 us (one
// tile per block, half of the CUs), and 5 us for the sum of the rows.
constexpr int kTrainRow = (kParams + 1 + 63) / 64 * 64;
constexpr uint32_t kTrainBlocks = 256;  // one per CU

// Place of (feature f of the 16 of tile ft, record r of the 16 of wave rt) in
// an LDS array of operands: 16x16 tiles, 4 records of a lane together.
__device__ __forceinline__ int train_frag(int ft, int rt, int f, int r) {
  return (ft * 4 + rt) * 256 + ((r >> 2) * 16 + f) * 4 + (r & 3);
}

// acc += the product of two operands over the 64 records.
__device__ __forceinline__ void train_outer(const h4 a[4], const h4 b[4], f4v& acc) {
#pragma unroll
  for (int kc = 0; kc < 4; kc++) acc = mfma16(a[kc], b[kc], acc);
}
__device__ __forceinline__ void train_operand(const _Float16* tile, int lane, h4 x[4]) {
#pragma unroll
  for (int kc = 0; kc < 4; kc++) x[kc] = *reinterpret_cast<const h4*>(tile + kc * 256 + 4 * lane);
}

__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
k_guide_train(GuideNet net, const TrainRecord* recs, const uint32_t* batch, uint32_t B, float wnorm, float wmax,
              float* partial) {
  __shared__ __align__(16) _Float16 sW[kWeights];
  __shared__ __align__(16) _Float16 sWt[kBackWeights];
  __shared__ float sB[kBiases];
  __shared__ __align__(16) _Float16 sAct[(kIn + 4 * kHid) * 64];  // layer inputs A_0..A_4 (train_frag)
  __shared__ __align__(16) _Float16 sDz[(4 * kHid + kOut) * 64];  // output gradients dZ_0..dZ_4 (train_frag)
  __shared__ float sLoss[4];
  constexpr int kOutStride = kOut + 1;
  float* const sOut = reinterpret_cast<float*>(sDz);  // raw outputs [record][output], in the place of dZ_0 and dZ_1
  static_assert(64 * kOutStride * 4 <= 2 * kHid * 64 * 2, "raw outputs overlap dZ_4");
  load_weights_lds_train(sW, sWt, sB, net.w, net.b);
  const int lane = __lane_id();
  const int v = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  auto act_tile = [&](int l, int ft) { return sAct + ((l == 0 ? 0 : kIn / 16 + (l - 1) * (kHid / 16)) + ft) * 1024; };
  auto dz_tile = [&](int l, int ft) { return sDz + (l * (kHid / 16) + ft) * 1024; };
  const h4 ones = h4{1, 1, 1, 1};
  const f4v zero = f4v{0.f, 0.f, 0.f, 0.f};
  // wave w's weight gradient tiles: layer 0 (to = w, ti = i), layers 1..4 (to = i, ti = w)
  f4v g0[5], gh[3][4], g4[3], gb[kLayers];
#pragma unroll
  for (int i = 0; i < 5; i++) g0[i] = gb[i] = zero;
#pragma unroll
  for (int i = 0; i < 12; i++) gh[i / 4][i % 4] = zero;
#pragma unroll
  for (int i = 0; i < 3; i++) g4[i] = zero;
  float loss = 0.f;
  const uint32_t tiles = (B + 63) / 64;
  for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const uint32_t ridx = tile * 64 + 16 * wave + v;
    const bool valid = ridx < B;
    TrainRecord rec{};
    if (valid) rec = recs[batch ? batch[ridx] : ridx];
    __syncthreads();  // weights loaded; the previous tile's operands read
    float f9[kFeat] = {rec.p[0], rec.p[1], rec.p[2], rec.n[0], rec.n[1], rec.n[2], rec.wi[0], rec.wi[1], rec.wi[2]};
    FeatScalars fs = feat_scalars(f9, net.lo, net.inv_ext);
    h4 act[4][4], xs[kIn / 16];
    {
      f4v out[3];
      forward_tile(sW, sB, fs, act, out, xs);
#pragma unroll
      for (int t = 0; t < 3; t++)
#pragma unroll
        for (int j = 0; j < 4; j++) sOut[(16 * wave + v) * kOutStride + 16 * t + 4 * g + j] = out[t][j];
    }
#pragma unroll
    for (int c = 0; c < kIn / 16; c++)
#pragma unroll
      for (int j = 0; j < 4; j++) act_tile(0, 0)[train_frag(c, wave, 4 * g + j, v)] = xs[c][j];
#pragma unroll
    for (int l = 0; l < 4; l++)
#pragma unroll
      for (int t = 0; t < 4; t++)
#pragma unroll
        for (int j = 0; j < 4; j++) act_tile(l + 1, 0)[train_frag(t, wave, 4 * g + j, v)] = act[l][t][j];
    __syncthreads();
    {
      const float* raw = sOut + (16 * wave + v) * kOutStride + 2 * kRawPerLobe * g;
      const bool used = valid && rec.w > 0.f;
      const float wn = fminf(rec.w * wnorm, wmax);
      float d[2 * kRawPerLobe];
      const float l = record_loss_grad(raw, mk(rec.dir[0], rec.dir[1], rec.dir[2]), wn, mk(rec.p[0], rec.p[1], rec.p[2]),
                                       mk(net.center[0], net.center[1], net.center[2]),
                                       mk(net.half[0], net.half[1], net.half[2]), d);
      if (used && g == 0) loss += l;
#pragma unroll
      for (int k = 0; k < 2 * kRawPerLobe; k++) {
        const int o = 2 * kRawPerLobe * g + k;
        dz_tile(4, 0)[train_frag(o >> 4, wave, o & 15, v)] = used ? (_Float16)(d[k] * kDzScale) : (_Float16)0.f;
      }
#pragma unroll
      for (int k = 0; k < (kOut - kLobes * kRawPerLobe) / 4; k++)  // padding outputs
        dz_tile(4, 0)[train_frag(2, wave, 8 + 2 * g + k, v)] = (_Float16)0.f;
    }
    __syncthreads();  // raw outputs read; dZ_4 written
    // backward through the hidden layers of this wave's 16 records
    h4 dz[4];  // dZ of the layer above, in B-operand form
#pragma unroll
    for (int l = 4; l >= 1; l--) {
      __builtin_amdgcn_sched_barrier(0);  // keep each layer's weight loads inside the layer
      f4v acc[4];
#pragma unroll
      for (int t = 0; t < 4; t++) acc[t] = zero;
#pragma unroll
      for (int c = 0; c < LayerOut(l) / 16; c++) {
        h4 b = dz[c];
        if (l == 4) {
#pragma unroll
          for (int j = 0; j < 4; j++) b[j] = dz_tile(4, 0)[train_frag(c, wave, 4 * g + j, v)];
        }
#pragma unroll
        for (int t = 0; t < 4; t++)
          acc[t] = mfma16(*reinterpret_cast<const h4*>(sWt + back_frag_base(l, t, c) + 4 * lane), b, acc[t]);
      }
#pragma unroll
      for (int t = 0; t < 4; t++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          _Float16 x = act[l - 1][t][j] > (_Float16)0.f ? (_Float16)acc[t][j] : (_Float16)0.f;
          dz[t][j] = x;
          dz_tile(l - 1, 0)[train_frag(t, wave, 4 * g + j, v)] = x;
        }
    }
    __syncthreads();
    // weight gradients: dW_l[out][in] = sum over the 64 records of dZ_l[out] A_l[in]
    h4 a[4], b[4];
    train_operand(dz_tile(0, wave), lane, a);
#pragma unroll
    for (int kc = 0; kc < 4; kc++) gb[0] = mfma16(a[kc], ones, gb[0]);
#pragma unroll
    for (int i = 0; i < 5; i++) {
      train_operand(act_tile(0, i), lane, b);
      train_outer(a, b, g0[i]);
    }
#pragma unroll
    for (int l = 1; l < kLayers; l++) {
      train_operand(act_tile(l, wave), lane, b);
#pragma unroll
      for (int i = 0; i < LayerOut(l) / 16; i++) {
        train_operand(dz_tile(l, i), lane, a);
        train_outer(a, b, l < 4 ? gh[l - 1][i] : g4[i]);
        if (i == wave) {
#pragma unroll
          for (int kc = 0; kc < 4; kc++) gb[l] = mfma16(a[kc], ones, gb[l]);
        }
      }
    }
  }
  float* const row = partial + size_t(blockIdx.x) * kTrainRow;
  auto put = [&](int l, int to, int ti, f4v x) {
#pragma unroll
    for (int j = 0; j < 4; j++)
      row[WeightOffset(l) + (16 * to + 4 * g + j) * LayerIn(l) + 16 * ti + v] = x[j] * (1.f / kDzScale);
  };
#pragma unroll
  for (int i = 0; i < 5; i++) put(0, wave, i, g0[i]);
#pragma unroll
  for (int l = 1; l < kLayers; l++)
#pragma unroll
    for (int i = 0; i < LayerOut(l) / 16; i++) put(l, i, wave, l < 4 ? gh[l - 1][i] : g4[i]);
#pragma unroll
  for (int l = 0; l < kLayers; l++)
    if (v == 0 && 16 * wave < LayerOut(l)) {
#pragma unroll
      for (int j = 0; j < 4; j++) row[BiasOffset(l) + 16 * wave + 4 * g + j] = gb[l][j] * (1.f / kDzScale);
    }
#pragma unroll
  for (int k = 32; k > 0; k >>= 1) loss += __shfl_xor(loss, k);
  if (lane == 0) sLoss[wave] = loss;
  __syncthreads();
  if (threadIdx.x == 0) row[kParams] = sLoss[0] + sLoss[1] + sLoss[2] + sLoss[3];
}

// grad += the sum of the partial rows, *loss += that of their losses.
__global__ void __launch_bounds__(256) k_guide_train_sum(const float* partial, uint32_t rows, float* grad, float* loss) {
  __shared__ float part[4][64];
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t i = blockIdx.x * 64 + lane;  // the rows are padded to a multiple of 64
  float s = 0.f;
#pragma unroll 8
  for (uint32_t r = wave; r < rows; r += 4) s += partial[size_t(r) * kTrainRow + i];
  part[wave][lane] = s;
  __syncthreads();
  if (wave != 0 || i > uint32_t(kParams)) return;
  s = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
  if (i < uint32_t(kParams))
    grad[i] += s;
  else
    *loss += s;
}

// Adam on the FP32 master weights; refreshes the FP16 / bias copies the
// kernels read and clears the gradient.
__global__ void k_guide_adam(float* p, float* grad, float* m1, float* m2, _Float16* wh, float* bias, float lr, float b1t,
                             float b2t, float gscale) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= kParams) return;
  const float b1 = 0.9f, b2 = 0.99f, eps = 1e-8f;
  float gi = grad[i] * gscale;
  float a = b1 * m1[i] + (1.f - b1) * gi;
  float c = b2 * m2[i] + (1.f - b2) * gi * gi;
  m1[i] = a;
  m2[i] = c;
  float x = p[i] - lr * (a / (1.f - b1t)) / (sqrtf(c / (1.f - b2t)) + eps);
  p[i] = x;
  grad[i] = 0.f;
  for (int l = 0; l < kLayers; l++) {
    if (i >= WeightOffset(l) && i < BiasOffset(l)) wh[HalfOffset(l) + (i - WeightOffset(l))] = (_Float16)x;
    if (i >= BiasOffset(l) && i < WeightOffset(l + 1)) bias[l * kHid + (i - BiasOffset(l))] = x;
  }
}

// FP32 master -> FP16 / bias copies (no update); clears kParams + 1 words of
// `clear` (a gradient and its loss), if given.
__global__ void k_guide_publish(const float* p, _Float16* wh, float* bias, float* clear) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (clear && i <= kParams) clear[i] = 0.f;
  if (i >= kParams) return;
  float x = p[i];
  for (int l = 0; l < kLayers; l++) {
    if (i >= WeightOffset(l) && i < BiasOffset(l)) wh[HalfOffset(l) + (i - WeightOffset(l))] = (_Float16)x;
    if (i >= BiasOffset(l) && i < WeightOffset(l + 1)) bias[l * kHid + (i - BiasOffset(l))] = x;
  }
}

// Mixture probes: pdf of directions, and samples, for raw output rows.
constexpr uint32_t kProbeBlock = 128;
__global__ void __launch_bounds__(kProbeBlock) k_guide_pdf(const float* raw, const float* dirs, uint32_t n, float* pdf) {
  __shared__ float4 km[kLobes * kProbeBlock];
  __shared__ float2 pw[kLobes * kProbeBlock];
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const Mixture m = lane_mixture(km, pw, threadIdx.x, kProbeBlock);
  decode(m, raw, splat(0.f), splat(0.f), splat(1.f));  // the means taken as directions
  pdf[i] = mixture_pdf(m, mk(dirs[3 * i], dirs[3 * i + 1], dirs[3 * i + 2]));
}
__global__ void __launch_bounds__(kProbeBlock) k_guide_sample(const float* raw, const float* xi, uint32_t n, float* out) {
  __shared__ float4 km[kLobes * kProbeBlock];
  __shared__ float2 pw[kLobes * kProbeBlock];
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const Mixture m = lane_mixture(km, pw, threadIdx.x, kProbeBlock);
  decode(m, raw, splat(0.f), splat(0.f), splat(1.f));
  f3 d = mixture_sample(m, xi[3 * i], xi[3 * i + 1], xi[3 * i + 2]);
  out[4 * i] = d.x;
  out[4 * i + 1] = d.y;
  out[4 * i + 2] = d.z;
  out[4 * i + 3] = mixture_pdf(m, d);
}

// Uniform random minibatch of record indices (with replacement).
__global__ void k_guide_batch(uint32_t* batch, uint32_t B, uint32_t n, uint32_t seed) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= B) return;
  batch[i] = mix32(mix32(seed) ^ (i * 0x9e3779b9u + 0x7f4a7c15u)) % n;
}

// ---------------------------------------------------------------- host state
void InitParams(std::vector<float>& p, uint32_t seed) {
  p.assign(kParams, 0.f);
  std::mt19937 rng(seed);
  for (int l = 0; l < kLayers; l++) {
    float lim = std::sqrt(6.f / float(LayerIn(l))) * (l == kLayers - 1 ? 0.1f : 1.f);
    std::uniform_real_distribution<float> U(-lim, lim);
    for (int i = 0; i < LayerIn(l) * LayerOut(l); i++) p[WeightOffset(l) + i] = U(rng);
  }
}

GuideState::GuideState() {
  params.alloc(kParams * 4);
  grad.alloc(kParams * 4);
  m1.alloc(kParams * 4);
  m2.alloc(kParams * 4);
  wh.alloc(kWeights * 2);
  bias.alloc(kBiases * 4);
  pub_wh.alloc(kWeights * 2);
  pub_bias.alloc(kBiases * 4);
  scal.alloc(64);
  std::vector<float> p;
  InitParams(p, 1234u);
  Upload(p);
}

void GuideState::Upload(const std::vector<float>& p) {
  if (p.size() != size_t(kParams)) throw std::runtime_error("guide parameter count mismatch");
  HipCheck(hipMemcpy(params.ptr, p.data(), kParams * 4, hipMemcpyHostToDevice), "guide params");
  HipCheck(hipMemset(grad.ptr, 0, kParams * 4), "guide grad");
  HipCheck(hipMemset(m1.ptr, 0, kParams * 4), "guide m1");
  HipCheck(hipMemset(m2.ptr, 0, kParams * 4), "guide m2");
  hipLaunchKernelGGL(k_guide_publish, dim3((kParams + 255) / 256), dim3(256), 0, nullptr, params.as<float>(), wh.as<_Float16>(),
                     bias.as<float>(), static_cast<float*>(nullptr));
  HipCheck(hipGetLastError(), "guide publish");
  HipCheck(hipDeviceSynchronize(), "guide publish");
  Publish(nullptr);
  steps = 0;
}

void GuideState::Publish(hipStream_t s) {
  HipCheck(hipStreamSynchronize(s), "guide training");
  std::lock_guard<std::mutex> lk(pub_mu);
  HipCheck(hipMemcpyAsync(pub_wh.ptr, wh.ptr, kWeights * 2, hipMemcpyDeviceToDevice, s), "publish guide weights");
  HipCheck(hipMemcpyAsync(pub_bias.ptr, bias.ptr, kBiases * 4, hipMemcpyDeviceToDevice, s), "publish guide biases");
  HipCheck(hipStreamSynchronize(s), "publish guide");
}

void GuideState::Snapshot(void* wh_dst, void* bias_dst) {
  std::lock_guard<std::mutex> lk(pub_mu);
  HipCheck(hipMemcpy(wh_dst, pub_wh.ptr, kWeights * 2, hipMemcpyDeviceToDevice), "guide snapshot");
  HipCheck(hipMemcpy(bias_dst, pub_bias.ptr, kBiases * 4, hipMemcpyDeviceToDevice), "guide snapshot");
}

static GuideNet MakeNet(const _Float16* w, const float* b, const float lo[3], const float hi[3], float alpha, float min_rough) {
  GuideNet n;
  n.w = w;
  n.b = b;
  for (int i = 0; i < 3; i++) {
    float e = hi[i] - lo[i];
    n.lo[i] = lo[i];
    n.inv_ext[i] = e > 0.f ? 1.f / e : 0.f;
  }
  for (int i = 0; i < 3; i++) {
    n.center[i] = 0.5f * (lo[i] + hi[i]);
    n.half[i] = std::max(0.5f * (hi[i] - lo[i]), 1e-6f);
  }
  n.alpha = alpha;
  n.min_rough = min_rough;
  n.max_depth = 0xffffffffu;
  return n;
}

GuideNet GuideState::Net(const float lo[3], const float hi[3], float alpha, float min_rough) const {
  return MakeNet(wh.as<_Float16>(), bias.as<float>(), lo, hi, alpha, min_rough);
}

void LaunchInfer(const GuideNet& net, const float* feats, const uint32_t* n_dev, uint32_t n_host, const uint32_t* slot_of,
                 _Float16* raw, int blocks, hipStream_t s) {
  hipLaunchKernelGGL(k_guide_infer, dim3(blocks), dim3(256), 0, s, net, feats, n_dev, n_host, slot_of, raw);
}

size_t TrainWorkBytes(uint32_t B) { return size_t(std::min((B + 63) / 64, kTrainBlocks)) * kTrainRow * 4; }

void LaunchTrain(const GuideNet& net, const TrainRecord* recs, const uint32_t* batch, uint32_t B, float wnorm, float wmax,
                 float* work, float* grad, float* loss, hipStream_t s) {
  if (B == 0) return;
  const uint32_t rows = std::min((B + 63) / 64, kTrainBlocks);
  hipLaunchKernelGGL(k_guide_train, dim3(rows), dim3(256), 0, s, net, recs, batch, B, wnorm, wmax, work);
  hipLaunchKernelGGL(k_guide_train_sum, dim3(kTrainRow / 64), dim3(256), 0, s, work, rows, grad, loss);
}

void GuideState::Step(float lr, float gscale, hipStream_t s) {
  steps++;
  float b1t = std::pow(0.9f, float(steps)), b2t = std::pow(0.99f, float(steps));
  hipLaunchKernelGGL(k_guide_adam, dim3((kParams + 255) / 256), dim3(256), 0, s, params.as<float>(), grad.as<float>(),
                     m1.as<float>(), m2.as<float>(), wh.as<_Float16>(), bias.as<float>(), lr, b1t, b2t, gscale);
}

void LaunchBatch(uint32_t* batch, uint32_t B, uint32_t n, uint32_t seed, hipStream_t s) {
  if (B && n) hipLaunchKernelGGL(k_guide_batch, dim3((B + 255) / 256), dim3(256), 0, s, batch, B, n, seed);
}

void LaunchPdf(const float* raw, const float* dirs, uint32_t n, float* pdf, hipStream_t s) {
  if (n) hipLaunchKernelGGL(k_guide_pdf, dim3((n + kProbeBlock - 1) / kProbeBlock), dim3(kProbeBlock), 0, s, raw, dirs, n, pdf);
}
void LaunchSample(const float* raw, const float* xi, uint32_t n, float* out, hipStream_t s) {
  if (n) hipLaunchKernelGGL(k_guide_sample, dim3((n + kProbeBlock - 1) / kProbeBlock), dim3(kProbeBlock), 0, s, raw, xi, n, out);
}

}  // namespace guide
}  // namespace rad

// ---------------------------------------------------------------- C ABI
namespace rad {
void SetLastError(const std::string& msg);
}

namespace {

using namespace rad;
using namespace rad::guide;

static_assert(sizeof(rad_guide_record) == sizeof(TrainRecord), "rad_guide_record must mirror TrainRecord");
static_assert(RAD_GUIDE_PARAMS == kParams && RAD_GUIDE_RAW == kOut && RAD_GUIDE_FEATS == kFeat, "guide ABI constants");

bool HaveDevice() {
  int count = 0;
  return hipGetDeviceCount(&count) == hipSuccess && count > 0;
}

template <class F>
rad_status Guarded(F&& f) {
  try {
    if (!HaveDevice()) {
      SetLastError("no HIP device available");
      return RAD_ERR_HIP;
    }
    f();
    return RAD_OK;
  } catch (const std::exception& e) {
    SetLastError(e.what());
    return RAD_ERR_HIP;
  }
}

// The network of one probe call, in one allocation with the call's own buffers:
// weights given by the caller.  (A GuideState draws random ones first, holds
// Adam's moments and a published copy, and allocates and clears each array by
// itself: a gradient of 32768 records took 403 us with one, now 220.)
struct ProbeNet {
  DeviceBuffer mem;
  GuideNet net;
  float* grad;     // kParams values and the loss, cleared
  char *in, *out;  // the call's buffers
  ProbeNet(const float* params, const float* bounds, size_t in_bytes, size_t out_bytes) {
    auto align = [](size_t v) { return (v + 255) & ~size_t(255); };
    const size_t sizes[] = {align(kParams * 4), align(kWeights * 2), align(kBiases * 4), align((kParams + 1) * 4), align(in_bytes)};
    size_t at[6] = {0};
    for (int i = 0; i < 5; i++) at[i + 1] = at[i] + sizes[i];
    mem.alloc(at[5] + align(out_bytes) + 256);
    char* const p = mem.as<char>();
    _Float16* const wh = reinterpret_cast<_Float16*>(p + at[1]);
    float* const bias = reinterpret_cast<float*>(p + at[2]);
    grad = reinterpret_cast<float*>(p + at[3]);
    in = p + at[4];
    out = p + at[5];
    HipCheck(hipMemcpy(p, params, kParams * 4, hipMemcpyHostToDevice), "guide params");
    hipLaunchKernelGGL(k_guide_publish, dim3(kParams / 256 + 1), dim3(256), 0, nullptr, reinterpret_cast<const float*>(p), wh, bias,
                       grad);
    HipCheck(hipGetLastError(), "guide publish");
    net = MakeNet(wh, bias, bounds, bounds + 3, 0.5f, 0.f);
  }
};

}  // namespace

extern "C" {

rad_status rad_hip_guide_forward(const float* params, const float* bounds, const float* feats, uint32_t n, float* raw) {
  if (!params || !bounds || (n && (!feats || !raw))) {
    SetLastError("NULL argument");
    return RAD_ERR_INVALID_ARG;
  }
  return Guarded([&] {
    ProbeNet p(params, bounds, size_t(n) * kFeat * 4, size_t(n) * kOut * 2);
    _Float16* const dr = reinterpret_cast<_Float16*>(p.out);
    HipCheck(hipMemcpy(p.in, feats, size_t(n) * kFeat * 4, hipMemcpyHostToDevice), "copy features");
    if (n)
      LaunchInfer(p.net, reinterpret_cast<const float*>(p.in), nullptr, n, nullptr, dr, std::min<uint32_t>(1024, (n + 63) / 64), nullptr);
    HipCheck(hipGetLastError(), "guide forward launch");
    std::vector<_Float16> h(size_t(n) * kOut);
    HipCheck(hipMemcpy(h.data(), dr, h.size() * 2, hipMemcpyDeviceToHost), "copy outputs");
    for (size_t i = 0; i < h.size(); i++) raw[i] = float(h[i]);
  });
}

rad_status rad_hip_guide_grad(const float* params, const float* bounds, const rad_guide_record* recs, uint32_t n,
                              float wnorm, float* grad, float* loss) {
  if (!params || !bounds || !grad || !loss || (n && !recs)) {
    SetLastError("NULL argument");
    return RAD_ERR_INVALID_ARG;
  }
  return Guarded([&] {
    ProbeNet p(params, bounds, size_t(n) * sizeof(TrainRecord), TrainWorkBytes(n));
    HipCheck(hipMemcpy(p.in, recs, size_t(n) * sizeof(TrainRecord), hipMemcpyHostToDevice), "copy records");
    LaunchTrain(p.net, reinterpret_cast<const TrainRecord*>(p.in), nullptr, n, wnorm, 64.f, reinterpret_cast<float*>(p.out), p.grad,
                p.grad + kParams, nullptr);
    HipCheck(hipGetLastError(), "guide train launch");
    std::vector<float> sums(kParams + 1);
    HipCheck(hipMemcpy(sums.data(), p.grad, sums.size() * 4, hipMemcpyDeviceToHost), "copy gradient");
    float inv = n ? 1.f / float(n) : 0.f;
    for (int i = 0; i < kParams; i++) grad[i] = sums[i] * inv;
    *loss = sums[kParams] * inv;
  });
}

rad_status rad_hip_guide_pdf(const float* raw, const float* dirs, uint32_t n, float* pdf) {
  if (!raw || (n && (!dirs || !pdf))) {
    SetLastError("NULL argument");
    return RAD_ERR_INVALID_ARG;
  }
  return Guarded([&] {
    DeviceBuffer dr, dd, dp;
    dr.alloc(kOut * 4);
    dd.alloc(std::max<size_t>(16, size_t(n) * 12));
    dp.alloc(std::max<size_t>(16, size_t(n) * 4));
    HipCheck(hipMemcpy(dr.ptr, raw, kRawPerLobe * kLobes * 4, hipMemcpyHostToDevice), "copy raw");
    HipCheck(hipMemcpy(dd.ptr, dirs, size_t(n) * 12, hipMemcpyHostToDevice), "copy dirs");
    LaunchPdf(dr.as<float>(), dd.as<float>(), n, dp.as<float>(), nullptr);
    HipCheck(hipGetLastError(), "guide pdf launch");
    HipCheck(hipMemcpy(pdf, dp.ptr, size_t(n) * 4, hipMemcpyDeviceToHost), "copy pdf");
  });
}

rad_status rad_hip_guide_sample(const float* raw, const float* xi, uint32_t n, float* out) {
  if (!raw || (n && (!xi || !out))) {
    SetLastError("NULL argument");
    return RAD_ERR_INVALID_ARG;
  }
  return Guarded([&] {
    DeviceBuffer dr, dx, dout;
    dr.alloc(kOut * 4);
    dx.alloc(std::max<size_t>(16, size_t(n) * 12));
    dout.alloc(std::max<size_t>(16, size_t(n) * 16));
    HipCheck(hipMemcpy(dr.ptr, raw, kRawPerLobe * kLobes * 4, hipMemcpyHostToDevice), "copy raw");
    HipCheck(hipMemcpy(dx.ptr, xi, size_t(n) * 12, hipMemcpyHostToDevice), "copy xi");
    LaunchSample(dr.as<float>(), dx.as<float>(), n, dout.as<float>(), nullptr);
    HipCheck(hipGetLastError(), "guide sample launch");
    HipCheck(hipMemcpy(out, dout.ptr, size_t(n) * 16, hipMemcpyDeviceToHost), "copy samples");
  });
}

rad_status rad_hip_scene_guide_get(rad_scene* scene, float* params, uint32_t* steps) {
  if (!scene || !params) {
    SetLastError("NULL argument");
    return RAD_ERR_INVALID_ARG;
  }
  return Guarded([&] {
    std::lock_guard<std::mutex> lk(scene->mu);
    HipCheck(hipSetDevice(scene->ctx->device), "hipSetDevice");
    if (!scene->guide) scene->guide = std::make_shared<GuideState>();
    HipCheck(hipMemcpy(params, scene->guide->params.ptr, kParams * 4, hipMemcpyDeviceToHost), "copy params");
    if (steps) *steps = scene->guide->steps;
  });
}

rad_status rad_hip_scene_guide_set(rad_scene* scene, const float* params) {
  if (!scene) {
    SetLastError("NULL argument");
    return RAD_ERR_INVALID_ARG;
  }
  return Guarded([&] {
    std::lock_guard<std::mutex> lk(scene->mu);
    HipCheck(hipSetDevice(scene->ctx->device), "hipSetDevice");
    if (!scene->guide) scene->guide = std::make_shared<GuideState>();
    std::vector<float> p;
    if (params)
      p.assign(params, params + kParams);
    else
      InitParams(p, 1234u);
    scene->guide->Upload(p);
  });
}

}  // extern "C"
