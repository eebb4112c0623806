// Fused multiply-adds and fixed-order sums of reduction partials (device code).
#pragma once
#include <hip/hip_runtime.h>

namespace bpx {
namespace {

__device__ inline double fmad(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ inline float fmad(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// Sum of partials[0..n) in a fixed order, by one wavefront: lane l folds
// l, l+64, ... into four accumulators (so its loads are in flight
// together), then an xor butterfly (each step adds the same two operands on
// both lanes of a pair, so every lane ends with the same bits). Every
// wavefront that folds the same partials gets the same value, whatever
// kernel or workgroup size it runs in.
__device__ inline double wave_fold(const double* __restrict__ part, int n) {
  const int lane = threadIdx.x & 63;
  double a0 = 0, a1 = 0, a2 = 0, a3 = 0;
  int i = lane;
  for (; i + 192 < n; i += 256) {
    a0 += part[i];
    a1 += part[i + 64];
    a2 += part[i + 128];
    a3 += part[i + 192];
  }
  for (; i < n; i += 64) a0 += part[i];
  double v = (a0 + a1) + (a2 + a3);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// wave_fold's value, its four accumulators formed by the first four
// wavefronts of a workgroup (for long lists), handed to every lane. s: 257
// doubles of LDS; ends with a barrier.
template <int NT>
__device__ inline double block_fold(const double* __restrict__ part, int n, double* s) {
  static_assert(NT >= 256, "four whole wavefronts");
  const int t = threadIdx.x;
  if (t < 256) {
    double a = 0;
    const int lane = t & 63, w = t >> 6;
    int base = lane;
    for (; base + 192 < n; base += 256) a += part[base + 64 * w];
    if (w == 0)
      for (; base < n; base += 64) a += part[base];
    s[t] = a;
  }
  __syncthreads();
  if (t < 64) {
    double v = (s[t] + s[t + 64]) + (s[t + 128] + s[t + 192]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if (t == 0) s[256] = v;
  }
  __syncthreads();
  return s[256];
}

// sum of v over a workgroup of NT lanes (64 or more) in a fixed order, in lane 0.
// s: NT doubles of LDS.
template <int NT>
__device__ inline double block_sum(double v, double* s) {
  const int t = threadIdx.x;
  __syncthreads();
  s[t] = v;
  __syncthreads();
  double a = 0;
  if (t < 64) {
#pragma unroll
    for (int i = 0; i < (NT + 63) / 64; ++i)
      if (t + 64 * i < NT) a += s[t + 64 * i];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) a += __shfl_xor(a, off, 64);
  }
  return a;
}

}  // namespace
}  // namespace bpx
