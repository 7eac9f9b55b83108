// Element access, operator application and reciprocals shared by the
// multigrid kernels (kernels_mg.hip, kernels_mgline.hip).
#pragma once
#include "mg.hpp"

namespace snac {
namespace {

template <typename T>
__device__ __forceinline__ long vidx(const MGLevT<T> &L, int m, int a, int s) { return ((long)m * L.na + a) * L.ns + s; }
template <typename T>
__device__ __forceinline__ long cidx(const MGLevT<T> &L, int m, int a, int s) { return m * L.qm + (long)a * L.ns + s; }

// sum of the couplings to the neighbouring lines (a and m directions) times x;
// wa, wm (a sweep on an odd periodic axis): row s of the line's entries of
// MGEnds, which take the place of x across the axis' ends
template <typename T>
__device__ __forceinline__ T nb_sum(const MGLevT<T> &L, const T *__restrict__ x, int m, int a, long e, long q,
                                    const T *wa = nullptr, const T *wm = nullptr) {
  T r = 0;
  const long sa = L.ns;
  if (a < L.na - 1) r += L.ca[q] * x[e + sa];
  else if (L.per_a) r += L.ca[q] * (wa ? wa[0] : x[e - (long)(L.na - 1) * sa]);
  if (a > 0) r += L.ca[q - sa] * x[e - sa];
  else if (L.per_a) r += L.ca[q + (long)(L.na - 1) * sa] * (wa ? wa[sa] : x[e + (long)(L.na - 1) * sa]);
  if (L.coupled) {
    const long sm = (long)L.na * L.ns;
    if (m < L.nm - 1) r += L.cm[q] * x[e + sm];
    else if (L.per_m) r += L.cm[q] * (wm ? wm[0] : x[e - (long)(L.nm - 1) * sm]);
    if (m > 0) r += L.cm[q - L.qm] * x[e - sm];
    else if (L.per_m) r += L.cm[q + (long)(L.nm - 1) * L.qm] * (wm ? wm[sa] : x[e + (long)(L.nm - 1) * sm]);
  }
  return r;
}

template <typename T>
__device__ __forceinline__ T mx_at(const MGLevT<T> &L, T lm, const T *__restrict__ x, int m, int a, int s) {
  const long e = vidx(L, m, a, s), q = cidx(L, m, a, s);
  T y = (L.dg[q] - lm * L.w[q]) * x[e];
  if (s > 0) y -= L.cs[q - 1] * x[e - 1];
  if (s < L.ns - 1) y -= L.cs[q] * x[e + 1];
  return y - nb_sum(L, x, m, a, e, q);
}

// Reciprocals for the relaxation's eliminations without the IEEE division
// sequence: the hardware estimate refined by Newton steps (two for FP64,
// one for FP32), within a few ulp of the correctly rounded quotient.  The
// relaxation only preconditions a CG that the FP64 residual judges.
__device__ __forceinline__ double frcp(double x) {
  double r = __builtin_amdgcn_rcp(x);
  double e = __builtin_fma(-x, r, 1.0);
  r = __builtin_fma(r, e, r);
  e = __builtin_fma(-x, r, 1.0);
  return __builtin_fma(r, e, r);
}
__device__ __forceinline__ float frcp(float x) {
  float r = __builtin_amdgcn_rcpf(x);
  float e = __builtin_fmaf(-x, r, 1.0f);
  return __builtin_fmaf(r, e, r);
}
// a / b, or a times the refined reciprocal of b (FR)
template <bool FR, typename T>
__device__ __forceinline__ T dv(T a, T b) {
  if constexpr (FR) return a * frcp(b);
  else return a / b;
}

}  // namespace
}  // namespace snac
