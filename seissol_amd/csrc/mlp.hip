// Training kernels of the friction warm-start MLP (6-32-32-1, tanh, FP32):
// mean-squared-error loss and gradient over a batch, Adam update, forward.
//
// A block takes kGroup (32) samples at a time, eight threads each: every thread
// has four of the 32 units of a layer, activations and deltas are exchanged
// through LDS, where the parameters are staged too, and then every thread sums
// its few weight gradients over the samples.  The sums stay in registers over
// the block's groups and go to the global gradient with one atomic per entry.
// Bound by the latency of the four dependent layers and by launches: 1024
// samples on 32 CUs instead of 8 (one sample per thread, all 32 units in turn),
// 50 -> 10 us; a whole training step 57 -> 13.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "engine.h"
#include "friction_common.h"

namespace sdg {
namespace friction {
namespace {

constexpr int kStride = kMlpInputs + 1;  // samples: features then target
constexpr int kGroup = 32, kPerSample = 8, kThreads = kGroup * kPerSample;
constexpr int kUnits = kMlpHidden / kPerSample;  // units of a layer per thread
constexpr int kLd = kMlpHidden + 1;              // padded row of 32 units
// Blocks: one per group up to one per CU, then as many as have eight groups
// each, up to four per CU: a block ends with 1,300 atomics, the same addresses
// for all (a step of 16,384 samples: 128 blocks 36 us, 256 38, 512 52; 131,072:
// 256 101, 512 86, 1024 107; 2 million: 256 1217, 512 773, 1024 631).
constexpr int64_t kMinFull = 256, kMaxBlocks = 1024, kGroupsPerBlock = 8;

__global__ void kZero(float* __restrict__ p, int n, float* __restrict__ loss) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.0f;
  if (i == 0) *loss = 0.0f;
}

__global__ __launch_bounds__(kThreads) void kLossGrad(const float* __restrict__ prm,
                                                      const float* __restrict__ samples, int64_t n,
                                                      float* __restrict__ grads, float* __restrict__ loss) {
  __shared__ float sP[kMlpParams];
  __shared__ float sW2[kMlpHidden * kLd];
  __shared__ float sX[kGroup * kStride];
  __shared__ float sZ[kGroup][kPerSample];
  __shared__ float sH1[kGroup][kLd], sD1[kGroup][kLd], sH2[kGroup][kLd], sD2[kGroup][kLd];
  __shared__ float sDy[kGroup];
  const int t = threadIdx.x, s = t / kPerSample, u = t % kPerSample, k0 = kUnits * u;
  for (int i = t; i < kMlpParams; i += kThreads) {
    const float v = prm[i];
    sP[i] = v;
    if (i >= kOffW2 && i < kOffB2) sW2[(i - kOffW2) / kMlpHidden * kLd + (i - kOffW2) % kMlpHidden] = v;
  }
  const float inv = 1.0f / static_cast<float>(n);
  float lossSum = 0.0f;
  // this thread's gradients: W2[gk][gj + 8 i], i < 4 (neighbouring threads add to
  // neighbouring entries: 16,384 samples 45 -> 38 us); W1[t / 6][t % 6] or, for the
  // last 64 threads, one of b1 and W3 (bk) or b2, and b3
  const int gk = t / kPerSample, gj = t % kPerSample;
  constexpr int kW1 = kMlpHidden * kMlpInputs;
  static_assert(kThreads == kW1 + 2 * kMlpHidden, "W1's entries, then two threads per unit");
  const int wk = t / kMlpInputs, wj = t % kMlpInputs, bk = (t - kW1) & (kMlpHidden - 1);
  float gW2[kUnits] = {}, g0 = 0.0f, g1 = 0.0f, g2 = 0.0f;

  for (int64_t first = static_cast<int64_t>(blockIdx.x) * kGroup; first < n;
       first += static_cast<int64_t>(gridDim.x) * kGroup) {
    const bool ok = first + s < n;
    __syncthreads();  // the previous group's sums have read everything
    if (t < kGroup * kStride) sX[t] = first * kStride + t < n * kStride ? samples[first * kStride + t] : 0.0f;
    __syncthreads();
    if (u < kMlpInputs) sZ[s][u] = ok ? (sX[s * kStride + u] - sP[kOffInMean + u]) / sP[kOffInScale + u] : 0.0f;
    __syncthreads();
    float h1[kUnits], h2[kUnits], d2[kUnits];
#pragma unroll
    for (int i = 0; i < kUnits; ++i) {
      float a = sP[kOffB1 + k0 + i];
#pragma unroll
      for (int j = 0; j < kMlpInputs; ++j) a += sP[kOffW1 + (k0 + i) * kMlpInputs + j] * sZ[s][j];
      h1[i] = tanhf(a);
      sH1[s][k0 + i] = ok ? h1[i] : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kUnits; ++i) h2[i] = sP[kOffB2 + k0 + i];
#pragma unroll 8
    for (int j = 0; j < kMlpHidden; ++j) {
      const float x = sH1[s][j];
#pragma unroll
      for (int i = 0; i < kUnits; ++i) h2[i] += sW2[(k0 + i) * kLd + j] * x;
    }
    float y = 0.0f;
#pragma unroll
    for (int i = 0; i < kUnits; ++i) {
      h2[i] = tanhf(h2[i]);
      sH2[s][k0 + i] = ok ? h2[i] : 0.0f;
      y += sP[kOffW3 + k0 + i] * h2[i];
    }
#pragma unroll
    for (int off = 1; off < kPerSample; off *= 2) y += __shfl_xor(y, off, 64);
    const float target = (sX[s * kStride + kMlpInputs] - sP[kOffOutMean]) / sP[kOffOutScale];
    const float r = ok ? sP[kOffB3] + y - target : 0.0f;
    const float dy = 2.0f * r * inv;
    if (u == 0) {
      sDy[s] = dy;
      lossSum += r * r * inv;
    }
#pragma unroll
    for (int i = 0; i < kUnits; ++i) {
      d2[i] = dy * sP[kOffW3 + k0 + i] * (1.0f - h2[i] * h2[i]);
      sD2[s][k0 + i] = d2[i];
    }
    __syncthreads();
    float d1[kUnits] = {};
#pragma unroll 8
    for (int k = 0; k < kMlpHidden; ++k) {
      const float x = sD2[s][k];
#pragma unroll
      for (int i = 0; i < kUnits; ++i) d1[i] += sW2[k * kLd + k0 + i] * x;
    }
#pragma unroll
    for (int i = 0; i < kUnits; ++i) sD1[s][k0 + i] = d1[i] * (1.0f - h1[i] * h1[i]);
    __syncthreads();
#pragma unroll 8
    for (int q = 0; q < kGroup; ++q) {
      const float x = sD2[q][gk];
#pragma unroll
      for (int i = 0; i < kUnits; ++i) gW2[i] += x * sH1[q][gj + kPerSample * i];
    }
    if (t < kW1) {
#pragma unroll 8
      for (int q = 0; q < kGroup; ++q) g0 += sD1[q][wk] * sZ[q][wj];
    } else if (t < kW1 + kMlpHidden) {
#pragma unroll 8
      for (int q = 0; q < kGroup; ++q) {
        g0 += sD1[q][bk];
        g1 += sDy[q] * sH2[q][bk];
        g2 += sDy[q];
      }
    } else {
#pragma unroll 8
      for (int q = 0; q < kGroup; ++q) g0 += sD2[q][bk];
    }
  }
#pragma unroll
  for (int i = 0; i < kUnits; ++i) atomicAdd(&grads[kOffW2 + gk * kMlpHidden + gj + kPerSample * i], gW2[i]);
  if (t < kW1) {
    atomicAdd(&grads[kOffW1 + t], g0);
  } else if (t < kW1 + kMlpHidden) {
    atomicAdd(&grads[kOffB1 + bk], g0);
    atomicAdd(&grads[kOffW3 + bk], g1);
    if (bk == 0) atomicAdd(&grads[kOffB3], g2);
  } else {
    atomicAdd(&grads[kOffB2 + bk], g0);
  }
  for (int off = 32; off > 0; off >>= 1) lossSum += __shfl_down(lossSum, off, 64);  // wave64 reduction
  if ((t & 63) == 0) atomicAdd(loss, lossSum);
}

__global__ void kAdam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                      float* __restrict__ v, float lr, float c1, float c2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < kOffW1 || i >= kMlpParams) return;  // normalisation constants are not trained
  const float beta1 = 0.9f, beta2 = 0.999f, eps = 1e-8f;
  const float gi = g[i];
  const float mi = beta1 * m[i] + (1.0f - beta1) * gi;
  const float vi = beta2 * v[i] + (1.0f - beta2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

__global__ void kForward(const float* __restrict__ prm, const float* __restrict__ x, int64_t n, int stride,
                         float* __restrict__ out) {
  __shared__ float sP[kMlpParams];
  for (int i = threadIdx.x; i < kMlpParams; i += blockDim.x) sP[i] = prm[i];
  __syncthreads();
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float f[kMlpInputs];
  for (int j = 0; j < kMlpInputs; ++j) f[j] = x[i * stride + j];
  out[i] = mlpEvaluate(sP, f);
}

}  // namespace
}  // namespace friction
}  // namespace sdg

using namespace sdg;

extern "C" {

int sdg_mlp_param_count(void) { return friction::kMlpParams; }

int sdg_mlp_loss_grad(const float* params, const float* samples, int64_t n, float* grads, float* loss, void* stream) {
  if (params == nullptr || samples == nullptr || grads == nullptr || loss == nullptr || n <= 0) {
    setError("sdg_mlp_loss_grad: invalid arguments");
    return SDG_ERR_INVALID;
  }
  auto st = static_cast<hipStream_t>(stream);
  friction::kZero<<<(friction::kMlpParams + 255) / 256, 256, 0, st>>>(grads, friction::kMlpParams, loss);
  const int64_t groups = (n + friction::kGroup - 1) / friction::kGroup;
  const int64_t full = std::clamp(groups / friction::kGroupsPerBlock, friction::kMinFull, friction::kMaxBlocks);
  const unsigned grid = static_cast<unsigned>(std::min(groups, full));
  friction::kLossGrad<<<grid, friction::kThreads, 0, st>>>(params, samples, n, grads, loss);
  SDG_HIP_CHECK(hipGetLastError());
  return SDG_OK;
}

int sdg_mlp_adam(float* params, const float* grads, float* m, float* v, int step, float lr, void* stream) {
  if (params == nullptr || grads == nullptr || m == nullptr || v == nullptr || step < 1) {
    setError("sdg_mlp_adam: invalid arguments");
    return SDG_ERR_INVALID;
  }
  const float c1 = 1.0f - powf(0.9f, static_cast<float>(step));
  const float c2 = 1.0f - powf(0.999f, static_cast<float>(step));
  friction::kAdam<<<(friction::kMlpParams + 255) / 256, 256, 0, static_cast<hipStream_t>(stream)>>>(
      params, grads, m, v, lr, c1, c2);
  SDG_HIP_CHECK(hipGetLastError());
  return SDG_OK;
}

int sdg_mlp_forward(const float* params, const float* features, int64_t n, int stride, float* out, void* stream) {
  if (params == nullptr || features == nullptr || out == nullptr || n < 0 || stride < friction::kMlpInputs) {
    setError("sdg_mlp_forward: invalid arguments");
    return SDG_ERR_INVALID;
  }
  if (n == 0) return SDG_OK;
  friction::kForward<<<static_cast<unsigned>((n + 255) / 256), 256, 0, static_cast<hipStream_t>(stream)>>>(
      params, features, n, stride, out);
  SDG_HIP_CHECK(hipGetLastError());
  return SDG_OK;
}

}  // extern "C"
