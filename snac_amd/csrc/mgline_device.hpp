// The factored lines' per-lane tables, rows and shapes (kernels_mgline.hip,
// kernels_mgpair.hip).
#pragma once
#include <stdexcept>
#include <type_traits>

#include "mg_device.hpp"

namespace snac {
namespace {

// ---- one line's factors, per lane ----
// Row j of a lane's K rows (1 <= j): D_j = G_j r_j - H_j D_{j-1} going down,
// D_j -= C_j D_{j+1} going up, x_j = D_j - A_j x_first - X_j x_last.
// Interface rows: first: r_0 - u0 D_1, last: D_last; NS reduction steps with
// the two multipliers of either row; then times the reciprocal diagonals.
// Rows and lanes that a line does not have are zeros throughout.
// FP32 (MODE 1, 2): D_j = (r_j - lo_j D_{j-1}) G_j with h = lo, and a division
// by i0, i1 in MODE 2: the unfactored kernels' operations in their order, with
// refined reciprocals (1) or IEEE quotients (2) in the table.
template <int K, int LPL, typename T>
struct LineFac {
  static constexpr int NS = LPL == 32 ? 6 : 7;
  static constexpr int NE = mg_fac_entries(K, LPL);
  T g[K - 1], h[K - 1], c[K - 1], a[K - 1], xq[K - 1], u0, k[4 * NS], i0, i1;
  __device__ __forceinline__ void load(const T *p) {
    int e = 0;
#pragma unroll
    for (int j = 0; j < K - 1; j++) g[j] = p[LPL * e++];
#pragma unroll
    for (int j = 0; j < K - 1; j++) h[j] = p[LPL * e++];
#pragma unroll
    for (int j = 0; j < K - 1; j++) c[j] = p[LPL * e++];
#pragma unroll
    for (int j = 0; j < K - 1; j++) a[j] = p[LPL * e++];
#pragma unroll
    for (int j = 0; j < K - 1; j++) xq[j] = p[LPL * e++];
    u0 = p[LPL * e++];
#pragma unroll
    for (int j = 0; j < 4 * NS; j++) k[j] = p[LPL * e++];
    i0 = p[LPL * e++];
    i1 = p[LPL * e++];
  }
};

__device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
template <typename T>
__device__ __forceinline__ T shf(T v, int src) { return __shfl(v, src, 64); }

// a lane's rows from / to memory: K contiguous values, as 16-byte pieces
// where every lane has all K (then they are 16-byte aligned)
template <int K, typename T, bool FULL>
__device__ __forceinline__ void rows_get(const T *p, int cnt, T (&v)[K]) {
  if constexpr (FULL && K * sizeof(T) % 16 == 0) {
    typedef T V __attribute__((ext_vector_type(16 / sizeof(T))));
    constexpr int W = 16 / sizeof(T);
#pragma unroll
    for (int q = 0; q < K / W; q++) {
      const V t = reinterpret_cast<const V *>(p)[q];
#pragma unroll
      for (int w = 0; w < W; w++) v[q * W + w] = t[w];
    }
  } else {
#pragma unroll
    for (int j = 0; j < K; j++) v[j] = FULL || j < cnt ? p[j] : T(0);
  }
}
template <int K, typename T, bool FULL>
__device__ __forceinline__ void rows_put(T *p, int cnt, const T (&v)[K]) {
  if constexpr (FULL && K * sizeof(T) % 16 == 0) {
    typedef T V __attribute__((ext_vector_type(16 / sizeof(T))));
    constexpr int W = 16 / sizeof(T);
#pragma unroll
    for (int q = 0; q < K / W; q++) {
      V t;
#pragma unroll
      for (int w = 0; w < W; w++) t[w] = v[q * W + w];
      reinterpret_cast<V *>(p)[q] = t;
    }
  } else {
#pragma unroll
    for (int j = 0; j < K; j++)
      if (FULL || j < cnt) p[j] = v[j];
  }
}

// the couplings of a column class to the columns above and below it
template <int K, int LPL, typename T>
__device__ __forceinline__ void coup_load(const T *p, T (&cap)[K], T (&cam)[K]) {
#pragma unroll
  for (int j = 0; j < K; j++) cap[j] = p[LPL * j];
#pragma unroll
  for (int j = 0; j < K; j++) cam[j] = p[LPL * (K + j)];
}

// calls go(K, LPL) as integral constants for the instance of a level
template <typename F>
void with_shape(int K, int lpl, F &&go) {
#define SNAC_SH(KK)                                                        \
  case KK:                                                                 \
    if (lpl == 32) go(std::integral_constant<int, KK>{}, std::integral_constant<int, 32>{}); \
    else go(std::integral_constant<int, KK>{}, std::integral_constant<int, 64>{});           \
    break;
  switch (K) {
    SNAC_SH(2) SNAC_SH(3) SNAC_SH(4) SNAC_SH(5) SNAC_SH(6) SNAC_SH(7) SNAC_SH(8)
    default: throw std::runtime_error("internal: no line-factor instance");
  }
#undef SNAC_SH
}

}  // namespace
}  // namespace snac
