// The learned-parameter network on the GPU: forward pass, mean-squared-error
// gradient and Adam update, parameters staged in LDS.
// Shape and parameter layout: csrc/host/learn.hpp (8 -> 32 -> 32 -> 2).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "launch.hpp"

namespace sc23ad::dev {
namespace {

constexpr int kIn = 8, kH = 32, kOut = 2;
constexpr int kOffW1 = 0, kOffB1 = kOffW1 + kH * kIn, kOffW2 = kOffB1 + kH,
              kOffB2 = kOffW2 + kH * kH, kOffW3 = kOffB2 + kH, kOffB3 = kOffW3 + kOut * kH,
              kNP = kOffB3 + kOut;
constexpr int kT = 256;
constexpr int kMaxParts = 128;  // workgroups of the gradient

__device__ __forceinline__ float sigm(float z) { return 1.0f / (1.0f + expf(-z)); }

struct Act {
  float h1[kH], h2[kH], y[kOut];
};

__device__ __forceinline__ void forward(const float* P, const float* x, Act& a) {
#pragma unroll 4
  for (int j = 0; j < kH; ++j) {
    float z = P[kOffB1 + j];
    for (int i = 0; i < kIn; ++i) z += P[kOffW1 + j * kIn + i] * x[i];
    a.h1[j] = tanhf(z);
  }
#pragma unroll 4
  for (int j = 0; j < kH; ++j) {
    float z = P[kOffB2 + j];
    for (int i = 0; i < kH; ++i) z += P[kOffW2 + j * kH + i] * a.h1[i];
    a.h2[j] = tanhf(z);
  }
  for (int k = 0; k < kOut; ++k) {
    float z = P[kOffB3 + k];
    for (int i = 0; i < kH; ++i) z += P[kOffW3 + k * kH + i] * a.h2[i];
    a.y[k] = sigm(z);
  }
}

__global__ __launch_bounds__(kT) void k_mlp_forward(int B, const float* __restrict__ X,
                                                    const float* __restrict__ Pg,
                                                    float* __restrict__ Y) {
  __shared__ float P[kNP];
  for (int k = threadIdx.x; k < kNP; k += kT) P[k] = Pg[k];
  __syncthreads();
  const int s = blockIdx.x * kT + threadIdx.x;
  if (s >= B) return;
  float x[kIn];
  for (int i = 0; i < kIn; ++i) x[i] = X[s * kIn + i];
  Act a;
  forward(P, x, a);
  for (int k = 0; k < kOut; ++k) Y[s * kOut + k] = a.y[k];
}

// Partial sums of (1/B) d/dP sum_s sum_k (y_sk - t_sk)^2 and of the loss over
// this workgroup's samples, to part[blockIdx.x * (kNP + 1) ...] (the loss last).
//
// The work is small (10 MFLOP at 1,220 samples) and was bound by LDS atomics:
// every sample added 1,410 values into one LDS array, 2,977 us.  Now a
// workgroup takes tiles of kS samples, 8 threads per sample for the forward
// and backward passes with the activations and their gradients in LDS, and
// each thread owns a few parameters, whose sums over the tile's samples it
// keeps in registers; k_mlp_reduce adds the workgroups in a fixed order.  Rows
// are padded to 36 floats (16-byte reads, rows on different banks).
constexpr int kS = 32, kRow = 36;
static_assert(kT == 8 * kS && kT == 8 * kH, "8 threads per sample, 8 per row of W2");

__global__ __launch_bounds__(kT) void k_mlp_grad(int B, const float* __restrict__ X,
                                                 const float* __restrict__ T,
                                                 const float* __restrict__ Pg,
                                                 float* __restrict__ part) {
  __shared__ float P[kNP];
  __shared__ __align__(16) float h1[kS][kRow], h2[kS][kRow], d1[kS][kRow], d2[kS][kRow];
  __shared__ float xs[kS][kIn + 1], d3[kS][kOut], ls[kS][kOut];
  const int t = threadIdx.x, s = t / 8, q = t % 8;
  constexpr int kU = kH / 8;  // hidden units per thread
  for (int k = t; k < kNP; k += kT) P[k] = Pg[k];
  const float inv_b = 1.0f / static_cast<float>(B);
  // this thread's parameters: W2[jr][4 q4 .. + 3], W1[jr][q4], and one of W3,
  // the biases and the loss
  const int jr = t / 8, q4 = t % 8;
  float g2[4] = {0, 0, 0, 0}, g1 = 0, gs = 0;
  for (int s0 = static_cast<int>(blockIdx.x) * kS; s0 < B; s0 += static_cast<int>(gridDim.x) * kS) {
    const int n = min(kS, B - s0);
    __syncthreads();
    if (t < kS * kIn) xs[t / kIn][t % kIn] = t / kIn < n ? X[s0 * kIn + t] : 0.0f;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int j = kU * q + u;
      float z = P[kOffB1 + j];
#pragma unroll
      for (int i = 0; i < kIn; ++i) z += P[kOffW1 + j * kIn + i] * xs[s][i];
      h1[s][j] = tanhf(z);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int j = kU * q + u;
      float z = P[kOffB2 + j];
#pragma unroll 8
      for (int i = 0; i < kH; ++i) z += P[kOffW2 + j * kH + i] * h1[s][i];
      h2[s][j] = tanhf(z);
    }
    __syncthreads();
    if (q < kOut) {
      float z = P[kOffB3 + q];
#pragma unroll 8
      for (int i = 0; i < kH; ++i) z += P[kOffW3 + q * kH + i] * h2[s][i];
      const float y = sigm(z);
      const float e = s < n ? y - T[(s0 + s) * kOut + q] : 0.0f;
      d3[s][q] = 2.0f * e * inv_b * y * (1.0f - y);  // zero past the last sample
      ls[s][q] = e * e * inv_b;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int i = kU * q + u;
      float acc = 0.0f;
#pragma unroll
      for (int k = 0; k < kOut; ++k) acc += P[kOffW3 + k * kH + i] * d3[s][k];
      d2[s][i] = acc * (1.0f - h2[s][i] * h2[s][i]);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int i = kU * q + u;
      float acc = 0.0f;
#pragma unroll 8
      for (int j = 0; j < kH; ++j) acc += P[kOffW2 + j * kH + i] * d2[s][j];
      d1[s][i] = acc * (1.0f - h1[s][i] * h1[s][i]);
    }
    __syncthreads();
#pragma unroll 8
    for (int r = 0; r < kS; ++r) {
      const float4 hv = *reinterpret_cast<const float4*>(&h1[r][4 * q4]);
      const float dv = d2[r][jr];
      g2[0] += dv * hv.x;
      g2[1] += dv * hv.y;
      g2[2] += dv * hv.z;
      g2[3] += dv * hv.w;
      g1 += d1[r][jr] * xs[r][q4];
    }
    if (t < kOut * kH) {
      for (int r = 0; r < kS; ++r) gs += d3[r][t / kH] * h2[r][t % kH];
    } else if (t < kOut * kH + kH) {
      for (int r = 0; r < kS; ++r) gs += d1[r][t - kOut * kH];
    } else if (t < kOut * kH + 2 * kH) {
      for (int r = 0; r < kS; ++r) gs += d2[r][t - kOut * kH - kH];
    } else if (t < kOut * kH + 2 * kH + kOut) {
      for (int r = 0; r < kS; ++r) gs += d3[r][t - kOut * kH - 2 * kH];
    } else if (t == kOut * kH + 2 * kH + kOut) {
      for (int r = 0; r < kS; ++r) gs += ls[r][0] + ls[r][1];
    }
  }
  float* out = part + static_cast<size_t>(blockIdx.x) * (kNP + 1);
#pragma unroll
  for (int u = 0; u < 4; ++u) out[kOffW2 + jr * kH + 4 * q4 + u] = g2[u];
  out[kOffW1 + jr * kIn + q4] = g1;
  if (t < kOut * kH) out[kOffW3 + t] = gs;
  else if (t < kOut * kH + kH) out[kOffB1 + t - kOut * kH] = gs;
  else if (t < kOut * kH + 2 * kH) out[kOffB2 + t - kOut * kH - kH] = gs;
  else if (t < kOut * kH + 2 * kH + kOut) out[kOffB3 + t - kOut * kH - 2 * kH] = gs;
  else if (t == kOut * kH + 2 * kH + kOut) out[kNP] = gs;
}

// G and *loss: the workgroups' partial sums, four interleaved chains each.
__global__ __launch_bounds__(kT) void k_mlp_reduce(int parts, const float* __restrict__ part,
                                                   float* __restrict__ G,
                                                   float* __restrict__ loss) {
  const int k = blockIdx.x * kT + threadIdx.x;
  if (k > kNP) return;
  float a[4] = {0, 0, 0, 0};
  int b = 0;
  for (; b + 4 <= parts; b += 4)
#pragma unroll
    for (int u = 0; u < 4; ++u) a[u] += part[static_cast<size_t>(b + u) * (kNP + 1) + k];
  for (; b < parts; ++b) a[0] += part[static_cast<size_t>(b) * (kNP + 1) + k];
  const float sum = (a[0] + a[1]) + (a[2] + a[3]);
  if (k < kNP) G[k] = sum;
  else *loss = sum;
}

__global__ __launch_bounds__(kT) void k_adam(int n, float* P, const float* G, float* M,
                                             float* V, float lr, float b1, float b2,
                                             float eps, float c1, float c2) {
  const int k = blockIdx.x * kT + threadIdx.x;
  if (k >= n) return;
  const float g = G[k];
  const float m = b1 * M[k] + (1.0f - b1) * g;
  const float v = b2 * V[k] + (1.0f - b2) * g * g;
  M[k] = m;
  V[k] = v;
  P[k] -= lr * (m / c1) / (sqrtf(v / c2) + eps);
}

}  // namespace

int mlp_param_count() { return kNP; }

hipError_t launch_mlp_forward(int B, const float* X, const float* P, float* Y, hipStream_t s) {
  if (B <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_mlp_forward, dim3((B + kT - 1) / kT), dim3(kT), 0, s, B, X, P, Y);
  return hipGetLastError();
}

size_t mlp_part_bytes() { return sizeof(float) * kMaxParts * (kNP + 1); }

hipError_t launch_mlp_grad(int B, const float* X, const float* T, const float* P, float* G,
                           float* loss, float* part, hipStream_t s) {
  const int parts = B > 0 ? static_cast<int>(std::min((static_cast<long long>(B) + kS - 1) / kS,
                                                      static_cast<long long>(kMaxParts)))
                          : 0;
  if (parts > 0) {
    hipLaunchKernelGGL(k_mlp_grad, dim3(parts), dim3(kT), 0, s, B, X, T, P, part);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k_mlp_reduce, dim3((kNP + kT) / kT), dim3(kT), 0, s, parts, part, G, loss);
  return hipGetLastError();
}

hipError_t launch_adam(int n, float* P, const float* G, float* M, float* V, float lr, int step,
                       hipStream_t s) {
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.0f - powf(b1, static_cast<float>(step));
  const float c2 = 1.0f - powf(b2, static_cast<float>(step));
  hipLaunchKernelGGL(k_adam, dim3((n + kT - 1) / kT), dim3(kT), 0, s, n, P, G, M, V, lr, b1, b2,
                     1e-8f, c1, c2);
  return hipGetLastError();
}

}  // namespace sc23ad::dev
