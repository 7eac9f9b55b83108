// Line relaxation of the FFT path's multigrid levels from precomputed
// factors (mg.hpp: MGFacT).  A line's tridiagonal system depends on its mode
// and on its column's coefficients, not on the solve, and most columns of a
// level share their coefficients (all of them on a uniform periodic axis; a
// handful of classes on a step).  The partitioned elimination of a line --
// Thomas within a lane's rows, parallel cyclic reduction of the two interface
// rows per lane -- is therefore factored once per (mode, class): what is left
// of a solve are the multiply-adds of the right-hand side, without divisions
// and with one number instead of a row of four through each shuffle.
//
// Bound: the sweeps by memory (b and x of half the lines, x of the other
// half) where a level is large, by the latency of one line's solve where it
// is small; the coarse end (k_tail_fac) by the chain of its line solves,
// about twenty in a row.  Measured per launch, unfactored and factored: the
// step's 48 modes, 512 x 80 in FP64, the sweeps over its four launched levels
// 11.4 -> 6.9 us on average, the coarse end 110 -> 42 us; the coarse end of 64
// modes, 128 rows in FP64 110 -> 36 us, of 64 modes, 256 rows in FP32 163 ->
// 75 us.  (Levels whose columns are all alike run kernels_mgpair.hip.)
#include "mgline_device.hpp"

namespace snac {
namespace {

// x of the calling lane's rows from their right-hand sides r (zero past cnt;
// FULL: every lane has K rows).  Lanes read only lanes of their own segment.
template <int K, int LPL, typename T, bool FULL, int MODE>
__device__ __forceinline__ void line_apply(const LineFac<K, LPL, T> &f, const T (&r)[K], int cnt, int lane, int seg0,
                                           T (&x)[K]) {
  T d[K];
  d[0] = r[0];
  d[1] = f.g[0] * r[1];
#pragma unroll
  for (int j = 2; j < K; j++)
    d[j] = MODE == 0 ? f.g[j - 1] * r[j] - f.h[j - 1] * d[j - 1] : (r[j] - f.h[j - 1] * d[j - 1]) * f.g[j - 1];
  T e1 = d[K - 1];
  if constexpr (!FULL && K > 2) e1 = cnt == K ? d[K - 1] : d[K - 2];
#pragma unroll
  for (int j = K - 3; j >= 1; j--) d[j] -= f.c[j - 1] * d[j + 1];
  T e0 = r[0] - f.u0 * d[1];
  {
    const T lo = shf(e1, seg0 + (lane > 0 ? lane - 1 : lane));
    const T hi = shf(e0, seg0 + (lane < LPL - 1 ? lane + 1 : lane));
    const T n0 = e0 - f.k[0] * lo - f.k[1] * e1;
    const T n1 = e1 - f.k[2] * e0 - f.k[3] * hi;
    e0 = n0;
    e1 = n1;
  }
#pragma unroll
  for (int q = 1, h = 1; h < LPL; q++, h <<= 1) {
    const int sm = seg0 + (lane >= h ? lane - h : lane), sp = seg0 + (lane + h < LPL ? lane + h : lane);
    const T a0 = shf(e0, sm), b0 = shf(e0, sp), a1 = shf(e1, sm), b1 = shf(e1, sp);
    e0 = e0 - f.k[4 * q] * a0 - f.k[4 * q + 1] * b0;
    e1 = e1 - f.k[4 * q + 2] * a1 - f.k[4 * q + 3] * b1;
  }
  const T xp = MODE == 2 ? e0 / f.i0 : e0 * f.i0, xl = MODE == 2 ? e1 / f.i1 : e1 * f.i1;
  x[0] = xp;
#pragma unroll
  for (int j = 1; j < K - 1; j++) x[j] = d[j] - f.a[j - 1] * xp - f.xq[j - 1] * xl;
  x[K - 1] = xl;
  if constexpr (!FULL && K > 2)
    if (cnt == K - 1) x[K - 2] = xl;
}

// One zebra colour of a launched level: a lane segment relaxes `lps`
// consecutive lines of one mode, its factors in registers (reloaded where
// the column class changes); the upper neighbour line of one line is the
// lower one of the next, and the next line's rows are loaded before this
// one is solved.  xc: neighbour lines are read with the prolongation of the
// next coarser level's xc added.
// WRAP: the colour with an odd periodic axis' ends a = 0 and na - 1, which
// are neighbours of one colour.  The segment of line 0 takes both: each
// reads the other's value from before the sweep (with xc0's prolongation,
// where a coarse correction came in between), so the sweep is a block Jacobi
// step within the colour and the same on every run.
template <int K, int LPL, typename T, bool FULL, bool WRAP, int MODE>
__global__ __launch_bounds__(256) void k_line_fac(MGLevT<T> L, MGFacT<T> F, T *__restrict__ x,
                                                  const T *__restrict__ b, int col, int nla, int zero_nb,
                                                  const int *__restrict__ done, const T *__restrict__ xc,
                                                  const T *__restrict__ xc0, int cna, int lps, int ngrp) {
  const int wl = threadIdx.x & 63, lane = wl & (LPL - 1), seg0 = wl - lane;
  const int sid = (int)(((long)blockIdx.x * 256 + threadIdx.x) / LPL);
  const int slot = sid / ngrp, grp = sid - slot * ngrp;
  if (slot >= *L.mcount) return;  // a whole lane segment leaves together
  const int m = L.mlist[slot];
  if (done && done[m]) return;
  const int na = L.na, ns = L.ns;
  const int p0 = FULL ? lane * K : lane * F.base + min(lane, F.extra);
  const int cnt = FULL ? K : (lane < F.nch ? F.base + (lane < F.extra ? 1 : 0) : 0);
  x += (long)m * na * ns + p0;
  b += (long)m * na * ns + p0;
  const long cm = (long)m * cna * ns + p0;
  const T *tab = F.tab + (long)m * F.ncls * LineFac<K, LPL, T>::NE * LPL + lane;
  auto nb = [&](int a, const T *c, T (&v)[K]) {
    rows_get<K, T, FULL>(x + (long)a * ns, cnt, v);
    if (c) {
      T w[K];
      rows_get<K, T, FULL>(c + cm + (long)(a >> 1) * ns, cnt, w);
#pragma unroll
      for (int j = 0; j < K; j++) v[j] += w[j];
    }
  };
  auto zero = [&](T (&v)[K]) {
#pragma unroll
    for (int j = 0; j < K; j++) v[j] = 0;
  };
  LineFac<K, LPL, T> f;
  T cap[K], cam[K];
  int cur = -1;
  auto factors = [&](int a) {
    const int c = F.ncls > 1 ? F.cls[a] : 0;
    if (c == cur) return;
    cur = c;
    f.load(tab + (long)c * LineFac<K, LPL, T>::NE * LPL);
    coup_load<K, LPL, T>(F.cc + (long)c * 2 * K * LPL + lane, cap, cam);
  };
  auto solve = [&](int a, const T (&bb)[K], const T (&vm)[K], const T (&vp)[K]) {
    T r[K], v[K];
#pragma unroll
    for (int j = 0; j < K; j++) r[j] = zero_nb ? bb[j] : bb[j] + fma_(cam[j], vm[j], cap[j] * vp[j]);
    line_apply<K, LPL, T, FULL, MODE>(f, r, cnt, lane, seg0, v);
    rows_put<K, T, FULL>(x + (long)a * ns, cnt, v);
  };
  const int nlw = WRAP ? nla - 1 : nla;  // the lines dealt out in groups
  const int j0 = grp * lps, j1 = min(j0 + lps, nlw);
  if (j0 >= j1) return;
  T vm[K], vp[K], bb[K], w0[K];
  zero(vm);
  zero(vp);
  int a = 2 * j0 + col;
  const bool wrap = WRAP && grp == 0 && !zero_nb;
  if (!zero_nb) {
    if (wrap) nb(0, xc0, w0);  // line 0 before this sweep
    if (a > 0 || L.per_a) nb(a > 0 ? a - 1 : na - 1, wrap ? xc0 : xc, vm);
    if (a < na - 1 || L.per_a) nb(a < na - 1 ? a + 1 : 0, xc, vp);
  }
  rows_get<K, T, FULL>(b + (long)a * ns, cnt, bb);
  for (int j = j0; j < j1; j++, a += 2) {
    factors(a);
    T nbb[K], nvp[K];
    zero(nvp);
    const bool more = j + 1 < j1;
    if (more) {
      rows_get<K, T, FULL>(b + (long)(a + 2) * ns, cnt, nbb);
      if (!zero_nb && (a + 2 < na - 1 || L.per_a)) nb(a + 2 < na - 1 ? a + 3 : 0, xc, nvp);
    }
    solve(a, bb, vm, vp);
    if (more) {
#pragma unroll
      for (int q = 0; q < K; q++) { vm[q] = vp[q]; vp[q] = nvp[q]; bb[q] = nbb[q]; }
    }
  }
  if (WRAP && grp == 0) {  // line na - 1
    a = na - 1;
    factors(a);
    zero(vm);
    if (!zero_nb) nb(a - 1, xc, vm);
    rows_get<K, T, FULL>(b + (long)a * ns, cnt, bb);
    if (zero_nb) zero(w0);
    solve(a, bb, vm, w0);
  }
}

// The coarse end of the V-cycle (MGTailT) for one mode per workgroup, with
// the levels' factors: as k_tail, one launch for all its levels, the mode's
// vectors in LDS (LX) or in memory.  After the colour-1 sweep only the
// colour-0 lines have a residual, the couplings to what was relaxed after
// them, so the FP64 restriction reads two lines of x per coarse line and
// nothing else.
template <int K, int LPL, typename T, bool LX, bool FULL, int MODE>
__global__ __launch_bounds__(512) void k_tail_fac(MGTailT<T> t, const T *__restrict__ lam,
                                                  const int *__restrict__ done) {
  extern __shared__ unsigned char smem_[];
  const int m = blockIdx.x;
  if (done && done[m]) return;
  T *lds = reinterpret_cast<T *>(smem_);
  const long mo = LX ? 0 : m;
  const T lmv = MODE != 0 ? lam[m] : T(0);
  auto X = [&](int l) -> T * { return LX ? lds + t.ox[l] : t.x[l] + mo * t.lev[l].na * t.lev[l].ns; };
  auto B = [&](int l) -> T * { return LX ? lds + t.ob[l] : t.b[l] + mo * t.lev[l].na * t.lev[l].ns; };
  const int ns = t.lev[0].ns;
  if (LX) {
    const int n0 = t.lev[0].na * ns;
    const T *bg = t.b[0] + (long)m * n0;
    for (int e = threadIdx.x; e < n0; e += 512) lds[t.ob[0] + e] = bg[e];
    __syncthreads();
  }
  constexpr int SEG = 512 / LPL;
  const int wl = threadIdx.x & 63, lane = wl & (LPL - 1), seg0 = wl - lane, seg = threadIdx.x / LPL;
  const MGFacT<T> &F0 = t.fac[0];
  const int p0 = FULL ? lane * K : lane * F0.base + min(lane, F0.extra);
  const int cnt = FULL ? K : (lane < F0.nch ? F0.base + (lane < F0.extra ? 1 : 0) : 0);
  LineFac<K, LPL, T> f;
  T cap[K], cam[K];
  int cl = -1, cc = -1;  // the level and class in registers
  auto factors = [&](int l, int a) {
    const MGFacT<T> &F = t.fac[l];
    const int c = F.ncls > 1 ? F.cls[a] : 0;
    if (l == cl && c == cc) return;
    cl = l;
    cc = c;
    f.load(F.tab + ((long)m * F.ncls + c) * LineFac<K, LPL, T>::NE * LPL + lane);
    coup_load<K, LPL, T>(F.cc + (long)c * 2 * K * LPL + lane, cap, cam);
  };
  // relaxes line a of level l; xc: the neighbours with the coarser level's
  // prolongation; wv: the value of a neighbour of the same colour (the ends
  // of an odd periodic axis) instead of what is stored
  auto relax = [&](int l, int a, bool zero_nb, const T *xc, const T *wv) {
    const int na = t.lev[l].na, per = t.lev[l].per_a;
    T *x = X(l) + p0;
    factors(l, a);
    T r[K], v[K];
    rows_get<K, T, FULL>(B(l) + a * ns + p0, cnt, r);
    if (!zero_nb) {
      T sum[K];
#pragma unroll
      for (int j = 0; j < K; j++) sum[j] = 0;
      auto add = [&](int an, bool same, const T (&w)[K]) {
        T nv[K];
        if (same && wv) {
#pragma unroll
          for (int j = 0; j < K; j++) nv[j] = wv[j];
        } else {
          rows_get<K, T, FULL>(x + an * ns, cnt, nv);
          if (xc) {
            T cv[K];
            rows_get<K, T, FULL>(xc + (an >> 1) * ns + p0, cnt, cv);
#pragma unroll
            for (int j = 0; j < K; j++) nv[j] += cv[j];
          }
        }
#pragma unroll
        for (int j = 0; j < K; j++) sum[j] = fma_(w[j], nv[j], sum[j]);
      };
      if (a < na - 1 || per) add(a < na - 1 ? a + 1 : 0, a == na - 1, cap);
      if (a > 0 || per) add(a > 0 ? a - 1 : na - 1, a == 0, cam);
#pragma unroll
      for (int j = 0; j < K; j++) r[j] += sum[j];
    }
    line_apply<K, LPL, T, FULL, MODE>(f, r, cnt, lane, seg0, v);
    rows_put<K, T, FULL>(x + a * ns, cnt, v);
  };
  for (int l = 0; l < t.nl - 1; l++) {
    const int na = t.lev[l].na, per = t.lev[l].per_a, nc = t.lev[l + 1].na;
    for (int c = 0; c < 2; c++) {
      for (int j = seg; 2 * j + c < na; j += SEG) relax(l, 2 * j + c, c == 0, nullptr, nullptr);
      __syncthreads();
    }
    const MGLevT<T> &L = t.lev[l];
    const T *x = X(l);
    T *bc = B(l + 1);
    for (int e = threadIdx.x; e < nc * ns; e += 512) {
      const int I = e / ns, s = e - I * ns, a = 2 * I;
      T r = 0;
      if (MODE != 0) {  // the residual as k_tail forms it
        for (int a2 = a; a2 <= a + 1 && a2 < na; a2++) {
          if (!L.act[cidx(L, 0, a2, s)]) continue;
          r += B(l)[vidx(L, 0, a2, s)] - mx_at(L, lmv, x, 0, a2, s);
        }
        bc[e] = r;
        continue;
      }
      if (a < na - 1 || per) r += L.ca[a * ns + s] * x[(a < na - 1 ? a + 1 : 0) * ns + s];
      if (a > 0 || per) r += L.ca[(a > 0 ? a - 1 : na - 1) * ns + s] * x[(a > 0 ? a - 1 : na - 1) * ns + s];
      bc[e] = r;
    }
    __syncthreads();
  }
  // the coarsest level's one line, with the pinned row of a singular mode
  // (its factors hold the identity row; the row's right-hand side is zero)
  {
    const int l = t.nl - 1;
    if (seg == 0) {
      factors(l, 0);
      T r[K], v[K];
      rows_get<K, T, FULL>(B(l) + p0, cnt, r);
      if (t.fac[l].pin && t.fac[l].pin[m]) {
#pragma unroll
        for (int j = 0; j < K; j++)
          if (p0 + j == t.fac[l].pin_s) r[j] = 0;
      }
      line_apply<K, LPL, T, FULL, MODE>(f, r, cnt, lane, seg0, v);
      rows_put<K, T, FULL>(X(l) + p0, cnt, v);
    }
    __syncthreads();
  }
  for (int l = t.nl - 2; l >= 0; l--) {
    const int na = t.lev[l].na;
    for (int j = seg; 2 * j + 1 < na; j += SEG) relax(l, 2 * j + 1, false, X(l + 1), nullptr);
    __syncthreads();
    // an odd periodic axis' ends are neighbours of one colour: segment 0
    // takes both, each with the other's value from before the sweep
    const bool wr = t.lev[l].per_a && (na & 1) && na > 1;
    const int nj = (na + 1) / 2 - (wr ? 1 : 0);
    T w0[K], w1[K];
    if (wr && seg == 0) {
      T cv[K];
      rows_get<K, T, FULL>(X(l) + p0, cnt, w0);
      rows_get<K, T, FULL>(X(l + 1) + p0, cnt, cv);
#pragma unroll
      for (int j = 0; j < K; j++) w0[j] += cv[j];
      rows_get<K, T, FULL>(X(l) + (na - 1) * ns + p0, cnt, w1);
      rows_get<K, T, FULL>(X(l + 1) + ((na - 1) >> 1) * ns + p0, cnt, cv);
#pragma unroll
      for (int j = 0; j < K; j++) w1[j] += cv[j];
    }
    for (int j = seg; j < nj; j += SEG) relax(l, 2 * j, false, nullptr, wr && j == 0 ? w1 : nullptr);
    if (wr && seg == 0) relax(l, na - 1, false, nullptr, w0);
    __syncthreads();
  }
  if (LX) {
    const int n0 = t.lev[0].na * ns;
    T *xg = t.x[0] + (long)m * n0;
    for (int e = threadIdx.x; e < n0; e += 512) xg[e] = lds[t.ox[0] + e];
  }
}

// coarse b = the restricted residual after a level's pre-smoothing from zero
// (colour 0 with its neighbours at zero, then colour 1): the colour-1 lines
// have none, a colour-0 line's is its couplings times the neighbours relaxed
// after it.  Rows across threads, RM modes per thread share the couplings.
// Bound by memory: half of x read (each line by two coarse lines, the second
// time from cache), half as much written; the general form reads b, all of x
// and five coefficients per row.  14.3 -> 6.0 us on average over the four
// launched levels of 64 modes, 512 columns, 128 rows.
__global__ __launch_bounds__(256) void k_restrict_zebra(MGLev F, int nc, const double *__restrict__ x,
                                                        double *__restrict__ bc, const int *__restrict__ done) {
  using T = double;
  constexpr int RM = 4;
  const int e = blockIdx.x * 256 + threadIdx.x, ns = F.ns, na = F.na;
  if (e >= nc * ns) return;
  const int I = e / ns, s = e - I * ns, a = 2 * I;
  const int live = *F.mcount;
  const bool hp = a < na - 1 || F.per_a, hm = a > 0 || F.per_a;
  const int ap = a < na - 1 ? a + 1 : 0, am = a > 0 ? a - 1 : na - 1;
  const T cp = hp ? F.ca[a * ns + s] : T(0), cm = hm ? F.ca[am * ns + s] : T(0);
  for (int q0 = blockIdx.y * RM; q0 < live; q0 += gridDim.y * RM) {
    T vp[RM], vm[RM];
    int md[RM];
#pragma unroll
    for (int k = 0; k < RM; k++) {
      md[k] = q0 + k < live ? F.mlist[q0 + k] : -1;
      if (md[k] >= 0 && done && done[md[k]]) md[k] = -1;
      const T *xm = x + (long)max(md[k], 0) * na * ns + s;
      vp[k] = hp && md[k] >= 0 ? xm[(long)ap * ns] : T(0);
      vm[k] = hm && md[k] >= 0 ? xm[(long)am * ns] : T(0);
    }
#pragma unroll
    for (int k = 0; k < RM; k++)
      if (md[k] >= 0) bc[(long)md[k] * nc * ns + e] = cp * vp[k] + cm * vm[k];
  }
}

// ---- the factorisation ----
template <typename T>
struct FacLev {
  const T *dg, *w, *cs;
  const int *rep;     // a column of each class
  const int *sing;    // singular modes with the row pin_s pinned (null: none)
  void *tab;
  int ns, ncls, nch, base, extra, pin_s;
};
constexpr int FAC_LEVS = 24;
template <typename T>
struct FacArgs {
  FacLev<T> lev[FAC_LEVS];
  const T *lam;
  int nm;
};

// One lane segment per (mode, class) of level blockIdx.y: the elimination of
// line_apply's comment carried out on the coefficients alone (MODE 1: with
// refined reciprocals).
template <int K, int LPL, typename T, int MODE>
__global__ __launch_bounds__(64) void k_line_factor(FacArgs<T> A) {
  const FacLev<T> &V = A.lev[blockIdx.y];
  const int lane = threadIdx.x & (LPL - 1), seg0 = threadIdx.x - lane;
  const int id = blockIdx.x * (64 / LPL) + threadIdx.x / LPL;
  if (id >= A.nm * V.ncls) return;
  const int m = id / V.ncls, c = id - m * V.ncls;
  const int cnt = lane < V.nch ? V.base + (lane < V.extra ? 1 : 0) : 0, p0 = lane * V.base + min(lane, V.extra);
  const long q0 = (long)V.rep[c] * V.ns;
  const T lam = A.lam[m];
  const bool pin = V.sing && V.sing[m];
  auto dv = [](T a, T b) -> T {
    if constexpr (MODE == 1) return a * frcp(b);
    else return a / b;
  };
  auto row = [&](int j, T &l, T &d, T &u) {
    const int s = p0 + j;
    d = V.dg[q0 + s] - lam * V.w[q0 + s];
    l = s > 0 ? -V.cs[q0 + s - 1] : T(0);
    u = s < V.ns - 1 ? -V.cs[q0 + s] : T(0);
    if (pin && s == V.pin_s) { d = 1; l = 0; u = 0; }
  };
  constexpr int NE = mg_fac_entries(K, LPL), R = K - 1;
  T *out = (T *)V.tab + (long)id * NE * LPL + lane;
  T G[K], H[K], C[K], Aa[K], X[K];
#pragma unroll
  for (int j = 0; j < K; j++) { G[j] = H[j] = C[j] = Aa[j] = X[j] = 0; }
  T aq = 0, cq = 0;
#pragma unroll
  for (int j = 1; j < K; j++) {
    if (j < cnt) {
      T l, d, u;
      row(j, l, d, u);
      G[j] = dv(T(1), j == 1 ? d : d - l * C[j - 1]);
      C[j] = u * G[j];
      if (j == 1) Aa[j] = l * G[j];
      else {
        Aa[j] = -l * Aa[j - 1] * G[j];
        H[j] = MODE == 0 ? l * G[j] : l;
      }
      if (j == cnt - 1) { aq = Aa[j]; cq = C[j]; }
    }
  }
  T CU[K];  // the couplings of the upward sweep (none on the last two rows)
#pragma unroll
  for (int j = 0; j < K; j++) CU[j] = j >= 1 && j <= cnt - 3 ? C[j] : T(0);
  T an = 0, cn = 0;
#pragma unroll
  for (int j = K - 2; j >= 1; j--) {
    if (j <= cnt - 2) {
      if (j == cnt - 2) { an = Aa[j]; cn = C[j]; }
      else { an = Aa[j] - C[j] * an; cn = -C[j] * cn; }
      Aa[j] = an;
      X[j] = cn;
    }
  }
  // interface rows (al, be, ga)
  T l0 = 0, d0 = 1, u0 = 0;
  if (cnt >= 2) row(0, l0, d0, u0);
  T al0 = 0, be0 = 1, ga0 = 0, al1 = 0, be1 = 1, ga1 = 0;
  if (cnt >= 2) {
    al0 = l0;
    be0 = cnt == 2 ? d0 : d0 - u0 * an;
    ga0 = cnt == 2 ? u0 : -u0 * cn;
    al1 = aq;
    ga1 = cq;
  }
  int e = 0;
  auto put = [&](T v) { out[LPL * e++] = v; };
  for (int j = 1; j <= R; j++) put(G[j]);
  for (int j = 1; j <= R; j++) put(H[j]);
  for (int j = 1; j <= R; j++) put(CU[j]);
  for (int j = 1; j <= R; j++) put(j <= cnt - 2 ? Aa[j] : T(0));
  for (int j = 1; j <= R; j++) put(j <= cnt - 2 ? X[j] : T(0));
  put(cnt > 2 ? u0 : T(0));
  auto sh = [&](T v, int src) { return __shfl(v, src, 64); };
  {
    const bool vm = lane > 0, vp = lane < LPL - 1;
    const int sm = seg0 + (vm ? lane - 1 : lane), sp = seg0 + (vp ? lane + 1 : lane);
    const T mal = sh(al1, sm), mbe = sh(be1, sm), mga = sh(ga1, sm);
    const T pal = sh(al0, sp), pbe = sh(be0, sp), pga = sh(ga0, sp);
    const T k1 = vm ? dv(al0, mbe) : T(0), k2 = dv(ga0, be1), k3 = dv(al1, be0), k4 = vp ? dv(ga1, pbe) : T(0);
    put(k1); put(k2); put(k3); put(k4);
    const T n0a = -k1 * mal, n0b = be0 - k1 * mga - k2 * al1, n0g = -k2 * ga1;
    const T n1a = -k3 * al0, n1b = be1 - k3 * ga0 - k4 * pal, n1g = -k4 * pga;
    al0 = n0a; be0 = n0b; ga0 = n0g;
    al1 = n1a; be1 = n1b; ga1 = n1g;
  }
  for (int h = 1; h < LPL; h <<= 1) {
    const bool vm = lane >= h, vp = lane + h < LPL;
    const int sm = seg0 + (vm ? lane - h : lane), sp = seg0 + (vp ? lane + h : lane);
    auto step = [&](T &al, T &be, T &ga) {
      const T mal = sh(al, sm), mbe = sh(be, sm), mga = sh(ga, sm);
      const T pal = sh(al, sp), pbe = sh(be, sp), pga = sh(ga, sp);
      const T k1 = vm ? dv(al, mbe) : T(0), k2 = vp ? dv(ga, pbe) : T(0);
      put(k1); put(k2);
      const T na = -k1 * mal, nb = be - k1 * mga - k2 * pal, ng = -k2 * pga;
      al = na; be = nb; ga = ng;
    };
    step(al0, be0, ga0);
    step(al1, be1, ga1);
  }
  // the reciprocal diagonals, or the diagonals to divide by
  put(MODE == 2 ? be0 : (cnt >= 2 ? dv(T(1), be0) : T(0)));
  put(MODE == 2 ? be1 : (cnt >= 2 ? dv(T(1), be1) : T(0)));
}

}  // namespace

// Lanes and rows per lane of the factored solves: 32 lanes (two lines per
// wavefront) while a lane's factors fit its registers beside the rows in
// flight -- FP64 up to 6 rows (192-row lines), FP32 up to 8 (256) -- else
// 64.  Longer chunks (and lines under four rows) keep the unfactored kernels.
template <typename T>
bool mg_fac_shape(int ns, MGFacT<T> &F) {
  if (ns < 4) return false;
  for (int lpl : {32, 64}) {
    const int nch = std::min(lpl, ns / 2), rows = (ns + nch - 1) / nch;
    const int K = rows;  // at least 2
    if (K > 8 || (lpl == 32 && sizeof(T) == 8 && K > 6)) continue;
    F.lpl = lpl;
    F.K = K;
    F.nch = nch;
    F.base = ns / nch;
    F.extra = ns % nch;
    return true;
  }
  return false;
}
template bool mg_fac_shape<double>(int, MGFacT<double> &);
template bool mg_fac_shape<float>(int, MGFacT<float> &);

template <typename T, int MODE>
void factor_levels(hipStream_t st, const MGHier<T> &H, int nm, const std::vector<size_t> &lev) {
  for (size_t q0 = 0; q0 < lev.size(); q0 += FAC_LEVS) {
    FacArgs<T> A;
    A.lam = H.lam;
    A.nm = nm;
    const int n = (int)std::min<size_t>(FAC_LEVS, lev.size() - q0);
    int mc = 1;
    for (int q = 0; q < n; q++) {
      const MGFacT<T> &F = H.fac[lev[q0 + q]];
      const MGLevT<T> &L = H.lev[lev[q0 + q]];
      A.lev[q] = FacLev<T>{L.dg, L.w, L.cs, F.rep, F.pin, (void *)F.tab, L.ns, F.ncls, F.nch, F.base, F.extra, F.pin_s};
      mc = std::max(mc, F.ncls);
    }
    // the line length, so the shape, is the same on every level
    with_shape(H.fac[lev[0]].K, H.fac[lev[0]].lpl, [&](auto kk, auto ll) {
      constexpr int K = decltype(kk)::value, LPL = decltype(ll)::value;
      const int per = 64 / LPL;
      hipLaunchKernelGGL((k_line_factor<K, LPL, T, MODE>), dim3((nm * mc + per - 1) / per, n), dim3(64), 0, st, A);
    });
    SNAC_HIP(hipGetLastError());
  }
}

template <typename T>
void mg_factor(hipStream_t st, const MGHier<T> &H, int nm, bool finest_only) {
  std::vector<size_t> lev[3];
  for (size_t l = 0; l < (finest_only ? 1 : H.fac.size()); l++)
    if (H.fac[l].tab) lev[H.fac[l].mode].push_back(l);
  if constexpr (sizeof(T) == 8) {
    factor_levels<T, 0>(st, H, nm, lev[0]);
  } else {
    factor_levels<T, 1>(st, H, nm, lev[1]);
    factor_levels<T, 2>(st, H, nm, lev[2]);
  }
}
template void mg_factor<double>(hipStream_t, const MGHier<double> &, int, bool);
template void mg_factor<float>(hipStream_t, const MGHier<float> &, int, bool);

template <typename T>
void mg_line_fac(hipStream_t st, const MGLevT<T> &L, const MGFacT<T> &F, T *x, const T *b, int col, int zero_nb,
                 const int *done, const T *xc, const T *xc0, int cna) {
  const int nla = (L.na - col + 1) / 2;
  if (nla <= 0) return;
  // lines per segment: as many as leave about eight wavefronts per CU (a
  // segment's factors are some forty loads, shared by its lines)
  const int spw = 64 / F.lpl;
  const int lps = (int)std::max<long>(1, std::min<long>(16, (long)nla * L.nm / (2048L * spw)));
  const bool wrap = col == 0 && L.per_a && (L.na & 1) && L.na > 1;
  const int nlw = wrap ? nla - 1 : nla, ngrp = (nlw + lps - 1) / lps;
  const long segs = (long)ngrp * L.nm;
  const dim3 grid((unsigned)((segs * F.lpl + 255) / 256));
  const bool full = L.ns == F.lpl * F.K;
  with_shape(F.K, F.lpl, [&](auto kk, auto ll) {
    constexpr int K = decltype(kk)::value, LPL = decltype(ll)::value;
#define SNAC_LF(FU, WR, MO)                                                                                    \
  hipLaunchKernelGGL((k_line_fac<K, LPL, T, FU, WR, MO>), grid, dim3(256), 0, st, L, F, x, b, col, nla, zero_nb, \
                     done, xc, xc0, cna, lps, ngrp)
    if constexpr (sizeof(T) == 8) {
      if (full) { if (wrap) SNAC_LF(true, true, 0); else SNAC_LF(true, false, 0); }
      else { if (wrap) SNAC_LF(false, true, 0); else SNAC_LF(false, false, 0); }
    } else {  // FP32 levels with an odd periodic axis are not factored
      if (F.mode == 1) { if (full) SNAC_LF(true, false, 1); else SNAC_LF(false, false, 1); }
      else { if (full) SNAC_LF(true, false, 2); else SNAC_LF(false, false, 2); }
    }
#undef SNAC_LF
  });
  SNAC_HIP(hipGetLastError());
}
template void mg_line_fac<double>(hipStream_t, const MGLevT<double> &, const MGFacT<double> &, double *, const double *,
                                  int, int, const int *, const double *, const double *, int);
template void mg_line_fac<float>(hipStream_t, const MGLevT<float> &, const MGFacT<float> &, float *, const float *, int,
                                 int, const int *, const float *, const float *, int);

template <typename T>
bool mg_tail_fac(hipStream_t st, const MGTailT<T> &t, int nm, const T *lam, const int *done) {
  constexpr int MODE = sizeof(T) == 8 ? 0 : 2;
  for (int l = 0; l < t.nl; l++)
    if (!t.fac[l].tab || t.fac[l].mode != MODE) return false;
  const MGFacT<T> &F = t.fac[0];
  const size_t shm = (size_t)t.lds_elems * sizeof(T);
  const bool lx = mg_tail_lds() && shm <= 160 * 1024, full = t.lev[0].ns == F.lpl * F.K;
  with_shape(F.K, F.lpl, [&](auto kk, auto ll) {
    constexpr int K = decltype(kk)::value, LPL = decltype(ll)::value;
#define SNAC_TF(LX, FU) \
  hipLaunchKernelGGL((k_tail_fac<K, LPL, T, LX, FU, MODE>), dim3(nm), dim3(512), LX ? shm : 0, st, t, lam, done)
    if (lx) { if (full) SNAC_TF(true, true); else SNAC_TF(true, false); }
    else { if (full) SNAC_TF(false, true); else SNAC_TF(false, false); }
#undef SNAC_TF
  });
  SNAC_HIP(hipGetLastError());
  return true;
}
template bool mg_tail_fac<double>(hipStream_t, const MGTailT<double> &, int, const double *, const int *);
template bool mg_tail_fac<float>(hipStream_t, const MGTailT<float> &, int, const float *, const int *);

void mg_restrict_zebra(hipStream_t st, const MGLev &F, const MGLev &C, const double *x, double *bc, const int *done) {
  const dim3 grid((unsigned)((C.na * C.ns + 255) / 256), (unsigned)((F.nm + 3) / 4));
  hipLaunchKernelGGL(k_restrict_zebra, grid, dim3(256), 0, st, F, C.na, x, bc, done);
  SNAC_HIP(hipGetLastError());
}

}  // namespace snac
