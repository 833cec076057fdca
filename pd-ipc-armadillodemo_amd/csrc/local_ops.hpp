// Rounding sequences of the local step and its residual, shared by the
// per-kernel path (k_local.hip, k_solve.hip) and the tile path (k_tiles.hip):
// every multiply-add that the compiler could contract in more than one way is
// spelled out, so both paths give the same bits.
#pragma once
#include <hip/hip_runtime.h>

namespace pdipc {

__device__ __forceinline__ double fmad(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fmad(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// a0^2 + a1^2 + a2^2
template <class T>
__device__ __forceinline__ T norm2(T a0, T a1, T a2) {
  return fmad(a2, a2, fmad(a0, a0, a1 * a1));
}

// c = (w^2 sum_j R1_ij b_j / D_j + (2 - w) w b_i) / D_i of one component, given
// the sum (PdIpcGpuFunc.cu:1041-1074)
__device__ __forceinline__ double first_term(double w, double sum, double b, double d) {
  return fmad(w * w, sum, (2.0 - w) * w * b) / d;
}

// First pass of the FP32-split residual M (M x) + c - x at one component: with
// y = M x = (1 - w) x + w (R1 x) / D and u = b / D, v = y + w u and the
// pointwise part (1 - w) y + (2 - w) w u - x
__device__ __forceinline__ void residual_first(double w, double x, double r1x, double b, double d, double* v,
                                               double* pt) {
  const double y = fmad(1.0 - w, x, w * r1x / d);
  const double u = b / d;
  *v = fmad(w, u, y);
  *pt = fmad((2.0 - w) * w, u, (1.0 - w) * y) - x;
}

// The rescale of a Laplace-Beltrami vector to the rest mean curvature h0
// (PdIpcGpuFunc.cu:668-707): a = sum_s L_s (x_s - x_i) (in T), lsum = sum_s L_s
template <class T>
__device__ __forceinline__ void curvature_rescale(const T (&a)[3], double lsum, const double (&xi)[3], double h0,
                                                  double (&out)[3]) {
#pragma unroll
  for (int k = 0; k < 3; k++) out[k] = fmad(lsum, xi[k], (double)a[k]);
  const double n = sqrt(norm2(out[0], out[1], out[2]));
  if (n >= 1e-10) {
    const double sc = h0 / n;
#pragma unroll
    for (int k = 0; k < 3; k++) out[k] *= sc;
  }
}

// One spring slot's force direction scaled: sp += stiff (rest / |d|) d
__device__ __forceinline__ float root(float x) { return sqrtf(x); }
__device__ __forceinline__ double root(double x) { return sqrt(x); }
template <class T>
__device__ __forceinline__ void add_spring(const T (&d)[3], double stiff, double rest, T (&sp)[3]) {
  const T len = root(norm2(d[0], d[1], d[2]));
  const T rc = (T)stiff * ((T)rest / len);
#pragma unroll
  for (int k = 0; k < 3; k++) sp[k] = fmad(rc, d[k], sp[k]);
}

// One workgroup of BT threads: the sum of n partials in a fixed order
template <int BT>
__device__ __forceinline__ void sum_partials(int n, const double* __restrict__ partials, double* __restrict__ out) {
  constexpr int kW = 64;
  __shared__ double red[BT / kW];
  double acc = 0.0;
  for (int i = threadIdx.x; i < n; i += BT) acc += partials[i];
  for (int off = kW / 2; off > 0; off >>= 1) acc += __shfl_down(acc, off, kW);
  if (threadIdx.x % kW == 0) red[threadIdx.x / kW] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < BT / kW; w++) t += red[w];
    *out = t;
  }
}

}  // namespace pdipc
