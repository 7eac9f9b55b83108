// Both colours of a multigrid level's zebra sweep in one launch (FFT path,
// factored lines), for the descent and for the ascent of the V-cycle.
//
// A lane segment marches over the level's line pairs (2I, 2I + 1): the
// colour-0 lines ahead of it, with their neighbours at zero, need nothing but
// b, so the colour-1 lines between them follow from registers.  On the way
// down that gives the residual that the next level starts from, the colour-0
// lines' couplings times the colour-1 lines, and nothing else is stored: on
// the way up the colour-0 lines are solved again from b, which costs less
// than keeping them, the colour-1 lines from these and the prolongation, and
// the colour-0 lines anew from those.  In vectors of the level: descent b
// read, a half written (one colour per launch and the restriction: 3.5);
// ascent b and half a vector read, one written (3.5).
// Bound by the chain of a segment's solves, so the independent lines of a
// step (the next colour-0 line, the colour-1 line, on the way up also the
// line to be stored) are solved together, two or three at a time.  64 modes,
// 512 columns, 128 rows: the finest level 19 us down, 27 us up (the memory's
// share is 8 and 13), the last launched one (64 columns) 7 and 8; five
// launches a level before, 8.9 us on average; a step 7.4 -> 6.0 ms.
// FP32 (64 modes, 256 x 256): the descent stores both colours for the
// restriction's own kernel, whose bits count, three launches a level: 12 us
// down, 18 up on the finest, 5 and 8 on the last launched (6.2 per colour
// before); a step 8.06 -> 7.67 ms.
// A segment solves the lines at its ends that its neighbours also solve, so
// no segment reads what another writes.
#include "mgline_device.hpp"

namespace snac {
namespace {

// line_apply for N lines of one class at once: the steps of a line's solve
// depend on each other, those of different lines overlap
template <int N, int K, int LPL, typename T, bool FULL, int MODE>
__device__ __forceinline__ void lines_apply(const LineFac<K, LPL, T> &f, const T (&r)[N][K], int cnt, int lane, int seg0,
                                            T (&x)[N][K]) {
  T d[N][K], e0[N], e1[N];
#pragma unroll
  for (int n = 0; n < N; n++) {
    d[n][0] = r[n][0];
    d[n][1] = f.g[0] * r[n][1];
  }
#pragma unroll
  for (int j = 2; j < K; j++)
#pragma unroll
    for (int n = 0; n < N; n++)
      d[n][j] = MODE == 0 ? f.g[j - 1] * r[n][j] - f.h[j - 1] * d[n][j - 1]
                          : (r[n][j] - f.h[j - 1] * d[n][j - 1]) * f.g[j - 1];
#pragma unroll
  for (int n = 0; n < N; n++) {
    e1[n] = d[n][K - 1];
    if constexpr (!FULL && K > 2) e1[n] = cnt == K ? d[n][K - 1] : d[n][K - 2];
  }
#pragma unroll
  for (int j = K - 3; j >= 1; j--)
#pragma unroll
    for (int n = 0; n < N; n++) d[n][j] -= f.c[j - 1] * d[n][j + 1];
#pragma unroll
  for (int n = 0; n < N; n++) e0[n] = r[n][0] - f.u0 * d[n][1];
  {
    const int sm = seg0 + (lane > 0 ? lane - 1 : lane), sp = seg0 + (lane < LPL - 1 ? lane + 1 : lane);
    T lo[N], hi[N];
#pragma unroll
    for (int n = 0; n < N; n++) {
      lo[n] = shf(e1[n], sm);
      hi[n] = shf(e0[n], sp);
    }
#pragma unroll
    for (int n = 0; n < N; n++) {
      const T n0 = e0[n] - f.k[0] * lo[n] - f.k[1] * e1[n];
      const T n1 = e1[n] - f.k[2] * e0[n] - f.k[3] * hi[n];
      e0[n] = n0;
      e1[n] = n1;
    }
  }
#pragma unroll
  for (int q = 1, h = 1; h < LPL; q++, h <<= 1) {
    const int sm = seg0 + (lane >= h ? lane - h : lane), sp = seg0 + (lane + h < LPL ? lane + h : lane);
    T a0[N], b0[N], a1[N], b1[N];
#pragma unroll
    for (int n = 0; n < N; n++) {
      a0[n] = shf(e0[n], sm);
      b0[n] = shf(e0[n], sp);
      a1[n] = shf(e1[n], sm);
      b1[n] = shf(e1[n], sp);
    }
#pragma unroll
    for (int n = 0; n < N; n++) {
      e0[n] = e0[n] - f.k[4 * q] * a0[n] - f.k[4 * q + 1] * b0[n];
      e1[n] = e1[n] - f.k[4 * q + 2] * a1[n] - f.k[4 * q + 3] * b1[n];
    }
  }
#pragma unroll
  for (int n = 0; n < N; n++) {
    const T xp = MODE == 2 ? e0[n] / f.i0 : e0[n] * f.i0, xl = MODE == 2 ? e1[n] / f.i1 : e1[n] * f.i1;
    x[n][0] = xp;
#pragma unroll
    for (int j = 1; j < K - 1; j++) x[n][j] = d[n][j] - f.a[j - 1] * xp - f.xq[j - 1] * xl;
    x[n][K - 1] = xl;
    if constexpr (!FULL && K > 2)
      if (cnt == K - 1) x[n][K - 2] = xl;
  }
}

// A segment's lines: positions u = 2 i0 - 2 ... 2 i1 of a periodic level.
template <int K, int LPL, typename T, bool FULL, int MODE>
struct March {
  LineFac<K, LPL, T> f;
  T cap[K], cam[K];
  const T *b;
  int m, i0, i1, lane, seg0, cnt, p0, na, ns;

  // false: no line for the calling thread's segment
  __device__ __forceinline__ bool init(const MGLevT<T> &L, const MGFacT<T> &F, const T *b_, const int *done,
                                       int nc, int r, int ngrp) {
    const int sid = (int)(((long)blockIdx.x * 256 + threadIdx.x) / LPL);
    const int slot = sid / ngrp, grp = sid - slot * ngrp;
    if (slot >= *L.mcount) return false;  // a whole lane segment leaves together
    m = L.mlist[slot];
    if (done && done[m]) return false;
    i0 = grp * r;
    i1 = min(i0 + r, nc);
    const int wl = threadIdx.x & 63;
    lane = wl & (LPL - 1);
    seg0 = wl - lane;
    p0 = FULL ? lane * K : lane * F.base + min(lane, F.extra);
    cnt = FULL ? K : (lane < F.nch ? F.base + (lane < F.extra ? 1 : 0) : 0);
    na = L.na;
    ns = L.ns;
    b = b_ + (long)m * na * ns + p0;
    f.load(F.tab + (long)m * LineFac<K, LPL, T>::NE * LPL + lane);
    coup_load<K, LPL, T>(F.cc + lane, cap, cam);
    return i0 < i1;
  }
  __device__ __forceinline__ int line(int u) const { return u < 0 ? u + na : u < na ? u : u - na; }
  // this lane's rows of b at u (on: else zeros)
  __device__ __forceinline__ void rows(int u, T (&v)[K], bool on = true) const {
    if (on) rows_get<K, T, FULL>(b + (long)line(u) * ns, cnt, v);
    else {
#pragma unroll
      for (int j = 0; j < K; j++) v[j] = 0;
    }
  }
  // adds the prolongation onto the colour-0 line at u (to the rounded value,
  // as if v came from memory: not fused with the product that v ends with)
  __device__ __forceinline__ void prolong(const T *c, int u, T (&v)[K]) const {
#pragma clang fp contract(off)
    T w[K];
    rows_get<K, T, FULL>(c + (long)(line(u) >> 1) * ns, cnt, w);
#pragma unroll
    for (int j = 0; j < K; j++) v[j] += w[j];
  }
  // x of N lines: right-hand sides b, plus the couplings to the lines below
  // (lo) and above (hi) unless bit n of Z says that there are none
  template <int Z, int N>
  __device__ __forceinline__ void solve(const T (&bb)[N][K], const T (&lo)[N][K], const T (&hi)[N][K],
                                        T (&x)[N][K]) const {
    T r[N][K];
#pragma unroll
    for (int n = 0; n < N; n++)
#pragma unroll
      for (int j = 0; j < K; j++)
        r[n][j] = (Z >> n) & 1 ? bb[n][j] : bb[n][j] + fma_(cam[j], lo[n][j], cap[j] * hi[n][j]);
    lines_apply<N, K, LPL, T, FULL, MODE>(f, r, cnt, lane, seg0, x);
  }
};

template <int K, typename T>
__device__ __forceinline__ void set(T (&d)[K], const T (&s)[K]) {
#pragma unroll
  for (int j = 0; j < K; j++) d[j] = s[j];
}

// The descent, colour 0 (neighbours at zero) and colour 1.  FP64: out = the
// restricted residual.  FP32: out = both colours, for a restriction of its
// own: the bits of the residual are those of the unfactored form.
template <int K, int LPL, typename T, bool FULL, int MODE>
__global__ __launch_bounds__(256) void k_pair_down(MGLevT<T> L, MGFacT<T> F, const T *__restrict__ b,
                                                   T *__restrict__ out, const int *__restrict__ done, int nc, int r,
                                                   int ngrp) {
  March<K, LPL, T, FULL, MODE> M;
  if (!M.init(L, F, b, done, nc, r, ngrp)) return;
  const int i0 = M.i0, i1 = M.i1, cnt = M.cnt;
  out += (long)M.m * (MODE == 0 ? nc : M.na) * M.ns + M.p0;
  T lo[2][K], hi[2][K], bb[2][K], nb[2][K], x[2][K], c[K], n[K], xm[K];
  if constexpr (MODE == 0) {
    M.rows(2 * i0 - 2, bb[0]);
    M.rows(2 * i0, bb[1]);
    M.rows(2 * i0 - 1, nb[0]);
    M.rows(2 * i0 + 2, nb[1]);
    M.template solve<3>(bb, lo, hi, x);
    set(lo[0], x[0]);
    set(hi[0], x[1]);
    set(c, x[1]);
  } else {
    M.rows(2 * i0, nb[0]);
    M.rows(2 * i0 + 2, nb[1]);
  }
  M.rows(2 * i0 + 1, bb[0]);
  M.rows(2 * i0 + 4, bb[1], i0 + 1 < i1);
  if constexpr (MODE == 0) {
    M.template solve<2>(nb, lo, hi, x);
    set(xm, x[0]);
  } else {
    M.template solve<3>(nb, lo, hi, x);
    set(c, x[0]);
  }
  set(n, x[1]);
  for (int I = i0; I < i1; I++) {
    const int u = 2 * I;
    T xp[K];
    if constexpr (MODE != 0) rows_put<K, T, FULL>(out + (long)u * M.ns, cnt, c);
    if (I + 1 < i1) {
      set(lo[0], c);
      set(hi[0], n);
      M.rows(u + 3, nb[0]);
      M.rows(u + 6, nb[1], I + 2 < i1);
      M.template solve<2>(bb, lo, hi, x);  // lines u + 1 and u + 4
      set(xp, x[0]);
      set(c, n);
      set(n, x[1]);
      set(bb[0], nb[0]);
      set(bb[1], nb[1]);
    } else {
      T l1[1][K], h1[1][K], b1[1][K], y[1][K];
      set(l1[0], c);
      set(h1[0], n);
      set(b1[0], bb[0]);
      M.template solve<0>(b1, l1, h1, y);
      set(xp, y[0]);
    }
    if constexpr (MODE == 0) {
      T v[K];
#pragma unroll
      for (int j = 0; j < K; j++) v[j] = M.cap[j] * xp[j] + M.cam[j] * xm[j];
      rows_put<K, T, FULL>(out + (long)I * M.ns, cnt, v);
      set(xm, xp);
    } else {
      rows_put<K, T, FULL>(out + (long)(u + 1) * M.ns, cnt, xp);
    }
  }
}

// The ascent: colour 1 against the colour-0 lines of the descent with xc
// added, then colour 0; x = both.
template <int K, int LPL, typename T, bool FULL, int MODE>
__global__ __launch_bounds__(256) void k_pair_up(MGLevT<T> L, MGFacT<T> F, T *__restrict__ x,
                                                 const T *__restrict__ b, const T *__restrict__ xc,
                                                 const int *__restrict__ done, int nc, int r, int ngrp) {
  March<K, LPL, T, FULL, MODE> M;
  if (!M.init(L, F, b, done, nc, r, ngrp)) return;
  const int i0 = M.i0, i1 = M.i1, cnt = M.cnt, ns = M.ns;
  x += (long)M.m * M.na * ns + M.p0;
  xc += (long)M.m * nc * ns + M.p0;
  T lo[3][K], hi[3][K], bb[3][K], nb[3][K], y[3][K], xm[K], xp[K], z1[K], z2[K];
  {
    const int u = 2 * i0;
    M.rows(u - 2, bb[0]);
    M.rows(u, bb[1]);
    M.rows(u + 2, bb[2]);
    M.rows(u - 1, nb[0]);
    M.rows(u + 1, nb[1]);
    M.rows(u + 4, nb[2], i0 + 1 < i1);
    M.template solve<7>(bb, lo, hi, y);
    M.prolong(xc, u - 2, y[0]);
    M.prolong(xc, u, y[1]);
    M.prolong(xc, u + 2, y[2]);
    set(lo[0], y[0]);
    set(hi[0], y[1]);
    set(lo[1], y[1]);
    set(hi[1], y[2]);
    set(z1, y[2]);
    set(bb[0], bb[1]);
    M.rows(u + 3, bb[1], i0 + 1 < i1);
    M.rows(u + 6, bb[2], i0 + 2 < i1);
    M.template solve<4>(nb, lo, hi, y);  // lines u - 1, u + 1 and u + 4
    if (i0 + 1 < i1) M.prolong(xc, u + 4, y[2]);
    set(xm, y[0]);
    set(xp, y[1]);
    set(z2, y[2]);
  }
  for (int I = i0; I < i1; I++) {
    const int u = 2 * I;
    if (I + 1 < i1) {
      set(lo[0], xm);
      set(hi[0], xp);
      set(lo[1], z1);
      set(hi[1], z2);
      const bool two = I + 2 < i1;
      M.rows(u + 2, nb[0]);
      M.rows(u + 5, nb[1], two);
      M.rows(u + 8, nb[2], I + 3 < i1);
      M.template solve<4>(bb, lo, hi, y);  // lines u, u + 3 and u + 6
      if (two) M.prolong(xc, u + 6, y[2]);
      rows_put<K, T, FULL>(x + (long)u * ns, cnt, y[0]);
      rows_put<K, T, FULL>(x + (long)(u + 1) * ns, cnt, xp);
      set(xm, xp);
      set(xp, y[1]);
      set(z1, z2);
      set(z2, y[2]);
#pragma unroll
      for (int n = 0; n < 3; n++) set(bb[n], nb[n]);
    } else {
      T l1[1][K], h1[1][K], b1[1][K], y1[1][K];
      set(l1[0], xm);
      set(h1[0], xp);
      set(b1[0], bb[0]);
      M.template solve<0>(b1, l1, h1, y1);
      rows_put<K, T, FULL>(x + (long)u * ns, cnt, y1[0]);
      rows_put<K, T, FULL>(x + (long)(u + 1) * ns, cnt, xp);
    }
  }
}

// shapes whose factors and lines in flight fit the registers of a wavefront
// or two per SIMD
template <typename T>
constexpr bool pair_instance(int K, int lpl) {
  return lpl == 32 ? (sizeof(T) == 4 || K <= 6) : (sizeof(T) == 8 && K <= 4);
}

// calls go(K, LPL, FULL, MODE) as integral constants for a level's instance
template <typename T, typename G>
void pair_shape(const MGLevT<T> &L, const MGFacT<T> &F, G &&go) {
  with_shape(F.K, F.lpl, [&](auto kk, auto ll) {
    constexpr int K = decltype(kk)::value, LPL = decltype(ll)::value;
    if constexpr (pair_instance<T>(K, LPL)) {
      auto mode = [&](auto full) {
        if constexpr (sizeof(T) == 8) go(kk, ll, full, std::integral_constant<int, 0>{});
        else if (F.mode == 1) go(kk, ll, full, std::integral_constant<int, 1>{});
        else go(kk, ll, full, std::integral_constant<int, 2>{});
      };
      if (L.ns == F.lpl * F.K) mode(std::true_type{});
      else mode(std::false_type{});
    } else {
      throw std::runtime_error("internal: no line-pair instance");
    }
  });
}

// Pairs per segment: as many as leave a wavefront per SIMD (of two that the
// registers allow).  A segment solves 2 r + 3 lines going down and 3 r + 3
// going up for its r pairs; a step of 64 modes, 512 columns, 128 rows with
// 512 / 1024 / 2048 / 4096 wavefronts: 6.3 / 6.0 / 6.1 / 6.2 ms.
template <typename T>
int pairs_per_segment(const MGLevT<T> &L, const MGFacT<T> &F, int nc) {
  return (int)std::max<long>(1, (long)nc * L.nm / (1024L * (64 / F.lpl)));
}

}  // namespace

// Levels whose columns are all alike (a uniform periodic axis of even
// length): 64 modes of 512 x 128 above; 256 modes of 512 x 256 in FP64 (64
// lanes) 36.5 -> 30.5 ms a step.  Where the columns fall into classes (a wall,
// a step) a segment reloads its factors at each class' end, and the launch
// waits for those segments: a step of 48 modes, 512 columns, 80 rows 10.4 ms
// against 9.3 with one colour per launch.
template <typename T>
bool mg_pair_fits(const MGLevT<T> &L, const MGFacT<T> &F) {
  return F.tab && F.ncls == 1 && pair_instance<T>(F.K, F.lpl) && !L.coupled && L.per_a && L.na >= 8 && L.na % 2 == 0;
}
template bool mg_pair_fits<double>(const MGLev &, const MGFacT<double> &);
template bool mg_pair_fits<float>(const MGLevT<float> &, const MGFacT<float> &);

template <typename T>
void mg_pair_down(hipStream_t st, const MGLevT<T> &L, const MGFacT<T> &F, const T *b, T *out, const int *done) {
  const int nc = L.na / 2, r = pairs_per_segment(L, F, nc), ngrp = (nc + r - 1) / r;
  const dim3 grid((unsigned)(((long)ngrp * L.nm * F.lpl + 255) / 256));
  pair_shape(L, F, [&](auto kk, auto ll, auto fu, auto mo) {
    hipLaunchKernelGGL((k_pair_down<decltype(kk)::value, decltype(ll)::value, T, decltype(fu)::value,
                                    decltype(mo)::value>),
                       grid, dim3(256), 0, st, L, F, b, out, done, nc, r, ngrp);
  });
  SNAC_HIP(hipGetLastError());
}
template void mg_pair_down<double>(hipStream_t, const MGLev &, const MGFacT<double> &, const double *, double *,
                                   const int *);
template void mg_pair_down<float>(hipStream_t, const MGLevT<float> &, const MGFacT<float> &, const float *, float *,
                                  const int *);

template <typename T>
void mg_pair_up(hipStream_t st, const MGLevT<T> &L, const MGFacT<T> &F, T *x, const T *b, const T *xc,
                const int *done) {
  const int nc = L.na / 2, r = pairs_per_segment(L, F, nc), ngrp = (nc + r - 1) / r;
  const dim3 grid((unsigned)(((long)ngrp * L.nm * F.lpl + 255) / 256));
  pair_shape(L, F, [&](auto kk, auto ll, auto fu, auto mo) {
    hipLaunchKernelGGL((k_pair_up<decltype(kk)::value, decltype(ll)::value, T, decltype(fu)::value,
                                  decltype(mo)::value>),
                       grid, dim3(256), 0, st, L, F, x, b, xc, done, nc, r, ngrp);
  });
  SNAC_HIP(hipGetLastError());
}
template void mg_pair_up<double>(hipStream_t, const MGLev &, const MGFacT<double> &, double *, const double *,
                                 const double *, const int *);
template void mg_pair_up<float>(hipStream_t, const MGLevT<float> &, const MGFacT<float> &, float *, const float *,
                                const float *, const int *);

}  // namespace snac
