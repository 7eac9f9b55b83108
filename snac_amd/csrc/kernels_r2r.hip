// Batched real-to-real transforms along one axis, the kinds FFTW offers and
// SNaC selects by boundary condition (fft.f90:96-149): R2HC/HC2R (periodic),
// REDFT10/REDFT01 (Neumann-Neumann), RODFT10/RODFT01 (Dirichlet-Dirichlet);
// REDFT11/RODFT11 (mixed), RODFT00 and lengths that are not powers of two are
// matrix products on the matrix cores.  Unnormalised, as FFTW's; callers
// scale.
//
// FFT path (n = 4..1024, powers of two): a workgroup stages L whole lines in
// LDS, forms the kind's n-point complex sequence (halfcomplex unpacking for
// HC2R, Makhoul's even/odd reordering for the cosine and sine kinds), and
// runs a two-pass Cooley-Tukey split n = N1*N2: every thread does one N1- or
// N2-point DFT entirely in registers, with one LDS transpose in between
// instead of log2(n) radix-2 stages through LDS.  Loads and stores walk the
// batch index with unit stride when the line stride is not 1, so a row of L
// neighbouring lines is one coalesced segment.
#include <cmath>
#include <map>
#include <mutex>
#include <vector>

#include "common.hpp"

namespace snac {
namespace {

constexpr int NT = 256;
constexpr int LDS_COMPLEX = 4096;  // complex doubles per workgroup (64 KiB)

enum { K_R2HC = 0, K_HC2R = 1, K_REDFT00 = 3, K_REDFT01 = 4, K_REDFT10 = 5, K_REDFT11 = 6, K_RODFT00 = 7,
       K_RODFT01 = 8, K_RODFT10 = 9, K_RODFT11 = 10 };

struct Args {
  const double *in;
  double *out;
  long ies, is1, is2, oes, os1, os2;
  int n, logn, nb1, nlines, L;
  int coal;  // 1: consecutive threads walk the batch index (line stride != 1)
  double scale;
  const double *tab;
  // lines of several fields in one launch (nlines counts them all): nf lines
  // each, field f at element offsets fin[f] / fout[f] from in / out
  int nf;
  long fin[R2R_FIELDS], fout[R2R_FIELDS];
};

// input and output offsets of a line (-1: past the last)
__device__ __forceinline__ void line_offset(const Args &a, int line, long &oi, long &oo) {
  oi = oo = -1;
  if (line >= a.nlines) return;
  int f = 0;
#pragma unroll
  for (int e = 1; e < R2R_FIELDS; e++) f += line >= e * a.nf;
  const int q = line - f * a.nf, b1 = q % a.nb1, b2 = q / a.nb1;
  oi = a.fin[f] + b1 * a.is1 + b2 * a.is2;
  oo = a.fout[f] + b1 * a.os1 + b2 * a.os2;
}

// lines per workgroup for an N1 x N2 FFT: one task per thread in each pass
// and at most LDS_COMPLEX complex values of LDS
constexpr int fft_lines(int n1, int n2) {
  return (NT / (n1 > n2 ? n1 : n2)) < (LDS_COMPLEX / (n1 * n2)) ? (NT / (n1 > n2 ? n1 : n2))
                                                                : (LDS_COMPLEX / (n1 * n2));
}

// Input / output offsets of the workgroup's L lines, one division each,
// kept in LDS so the per-element address is one multiply-add (-1: past the
// last line).  Ends with a barrier.
template <int L>
__device__ __forceinline__ void line_offsets(const Args &a, int line0, long (&oin)[L], long (&oout)[L]) {
  for (int t = threadIdx.x; t < L; t += NT) {
    const int line = line0 + t;
    long oi, oo;
    line_offset(a, line, oi, oo);
    oin[t] = oi;
    oout[t] = oo;
  }
  __syncthreads();
}

__device__ __forceinline__ void elem_of(const Args &a, int e, int &line, int &q) {
  if (a.coal) { line = e % a.L; q = e / a.L; }
  else { q = e % a.n; line = e / a.n; }
}

// radix-2 DIT on N values held in registers (fully unrolled; twiddle
// indices are compile-time, so the loads are uniform across the wavefront).
// tw[m] = e^{-2 pi i m/n}; stride = n/N maps W_N^m onto that table.
template <int N>
__device__ __forceinline__ void fft_reg(double2 (&v)[N], const double2 *__restrict__ tw, int stride, bool inv) {
  constexpr int LOG = (N >= 2) + (N >= 4) + (N >= 8) + (N >= 16) + (N >= 32);
#pragma unroll
  for (int i = 0; i < N; i++) {
    int j = 0;
#pragma unroll
    for (int b = 0; b < LOG; b++) j |= ((i >> b) & 1) << (LOG - 1 - b);
    if (j > i) { double2 t = v[i]; v[i] = v[j]; v[j] = t; }
  }
#pragma unroll
  for (int len = 2; len <= N; len <<= 1) {
#pragma unroll
    for (int i = 0; i < N; i += len) {
#pragma unroll
      for (int j = 0; j < len / 2; j++) {
        double2 w = tw[j * (N / len) * stride];
        if (inv) w.y = -w.y;
        double2 x0 = v[i + j], x1 = v[i + j + len / 2];
        double2 c = make_double2(x1.x * w.x - x1.y * w.y, x1.x * w.y + x1.y * w.x);
        v[i + j] = make_double2(x0.x + c.x, x0.y + c.y);
        v[i + j + len / 2] = make_double2(x0.x - c.x, x0.y - c.y);
      }
    }
  }
}

// R-point DFT in registers for the odd factors of the mixed-radix lengths
// (y_q = sum_r x_r e^{-2 pi i r q/R}, conjugated when inv)
template <int R>
__device__ __forceinline__ void dft_prime(double2 (&x)[R], bool inv) {
  const double sg = inv ? -1.0 : 1.0;
  if constexpr (R == 2) {
    const double2 a = x[0], b = x[1];
    x[0] = make_double2(a.x + b.x, a.y + b.y);
    x[1] = make_double2(a.x - b.x, a.y - b.y);
  } else if constexpr (R == 3) {
    const double s3 = sg * 0.86602540378443864676;  // sin(2 pi/3)
    const double2 t = make_double2(x[1].x + x[2].x, x[1].y + x[2].y);
    const double2 d = make_double2(s3 * (x[1].x - x[2].x), s3 * (x[1].y - x[2].y));
    const double2 m = make_double2(x[0].x - 0.5 * t.x, x[0].y - 0.5 * t.y);
    x[0] = make_double2(x[0].x + t.x, x[0].y + t.y);
    x[1] = make_double2(m.x + d.y, m.y - d.x);
    x[2] = make_double2(m.x - d.y, m.y + d.x);
  } else {
    static_assert(R == 5, "factors 2, 3 and 5");
    const double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;        // cos(2 pi/5), cos(4 pi/5)
    const double s1 = sg * 0.95105651629515357212, s2 = sg * 0.58778525229247312917;  // sin(2 pi/5), sin(4 pi/5)
    const double2 p1 = make_double2(x[1].x + x[4].x, x[1].y + x[4].y), q1 = make_double2(x[1].x - x[4].x, x[1].y - x[4].y);
    const double2 p2 = make_double2(x[2].x + x[3].x, x[2].y + x[3].y), q2 = make_double2(x[2].x - x[3].x, x[2].y - x[3].y);
    const double2 m1 = make_double2(x[0].x + c1 * p1.x + c2 * p2.x, x[0].y + c1 * p1.y + c2 * p2.y);
    const double2 m2 = make_double2(x[0].x + c2 * p1.x + c1 * p2.x, x[0].y + c2 * p1.y + c1 * p2.y);
    const double2 d1 = make_double2(s1 * q1.x + s2 * q2.x, s1 * q1.y + s2 * q2.y);
    const double2 d2 = make_double2(s2 * q1.x - s1 * q2.x, s2 * q1.y - s1 * q2.y);
    x[0] = make_double2(x[0].x + p1.x + p2.x, x[0].y + p1.y + p2.y);
    x[1] = make_double2(m1.x + d1.y, m1.y - d1.x);
    x[4] = make_double2(m1.x - d1.y, m1.y + d1.x);
    x[2] = make_double2(m2.x + d2.y, m2.y - d2.x);
    x[3] = make_double2(m2.x - d2.y, m2.y + d2.x);
  }
}
// N points of v, S apart from element O on, transformed into out (natural
// order): N = R M, M-point transforms of every R-th point, twiddles, R-point
// transforms across them.  Everything unrolls to registers; tw as in fft_reg.
template <int N, int O, int S, int NV>
__device__ __forceinline__ void dft_mixed(const double2 (&v)[NV], double2 (&out)[N], const double2 *__restrict__ tw,
                                          int stride, bool inv) {
  if constexpr (N == 1) {
    out[0] = v[O];
  } else {
    constexpr int R = N % 5 == 0 ? 5 : (N % 3 == 0 ? 3 : 2), M = N / R;
    double2 part[R][M];
    if constexpr (R >= 2) {
      dft_mixed<M, O, S * R, NV>(v, part[0], tw, stride * R, inv);
      dft_mixed<M, O + S, S * R, NV>(v, part[1], tw, stride * R, inv);
    }
    if constexpr (R >= 3) dft_mixed<M, O + 2 * S, S * R, NV>(v, part[2], tw, stride * R, inv);
    if constexpr (R >= 5) {
      dft_mixed<M, O + 3 * S, S * R, NV>(v, part[3], tw, stride * R, inv);
      dft_mixed<M, O + 4 * S, S * R, NV>(v, part[4], tw, stride * R, inv);
    }
#pragma unroll
    for (int k = 0; k < M; k++) {
      double2 x[R];
#pragma unroll
      for (int r = 0; r < R; r++) {
        x[r] = part[r][k];
        if (r * k != 0) {
          double2 w = tw[r * k * stride];
          if (inv) w.y = -w.y;
          x[r] = make_double2(part[r][k].x * w.x - part[r][k].y * w.y, part[r][k].x * w.y + part[r][k].y * w.x);
        }
      }
      dft_prime<R>(x, inv);
#pragma unroll
      for (int q = 0; q < R; q++) out[k + M * q] = x[q];
    }
  }
}
// the register DFT of either kind of length, in place
template <int N>
__device__ __forceinline__ void fft_any(double2 (&v)[N], const double2 *__restrict__ tw, int stride, bool inv) {
  if constexpr ((N & (N - 1)) == 0) {
    fft_reg<N>(v, tw, stride, inv);
  } else {
    double2 out[N];
    dft_mixed<N, 0, 1, N>(v, out, tw, stride, inv);
#pragma unroll
    for (int i = 0; i < N; i++) v[i] = out[i];
  }
}

// complex input slot s of the n-point sequence for KIND, from the raw line r
// (raw index n maps to zero where the kind needs x_n).  tk[k] = (cos, sin)(pi k / 2n).
template <int KIND>
__device__ __forceinline__ double2 pre_slot(const double *r, int s, int n, const double2 *tk) {
  const int h = n >> 1;
  if (KIND == K_R2HC) return make_double2(r[s], 0.0);
  if (KIND == K_HC2R) {
    if (s == 0 || s == h) return make_double2(r[s], 0.0);
    if (s < h) return make_double2(r[s], r[n - s]);
    return make_double2(r[n - s], -r[s]);
  }
  if (KIND == K_REDFT10 || KIND == K_RODFT10) {
    int q = (s < h) ? 2 * s : 2 * (n - 1 - s) + 1;
    double x = r[q];
    if (KIND == K_RODFT10 && (q & 1)) x = -x;
    return make_double2(x, 0.0);
  }
  // REDFT01 / RODFT01: e^{i pi s/(2n)} (a - i b)
  double a, b;
  if (KIND == K_REDFT01) { a = r[s]; b = (s == 0) ? 0.0 : r[n - s]; }
  else { a = r[n - 1 - s]; b = (s == 0) ? 0.0 : r[s - 1]; }
  double2 t = tk[s];
  return make_double2(a * t.x + b * t.y, a * t.y - b * t.x);
}

template <int KIND>
__device__ __forceinline__ double post_val(const double2 *z, int q, int n, const double2 *tk) {
  if (KIND == K_R2HC) return (q <= (n >> 1)) ? z[q].x : z[n - q].y;
  if (KIND == K_HC2R) return z[q].x;
  if (KIND == K_REDFT10 || KIND == K_RODFT10) {
    int k = (KIND == K_RODFT10) ? n - 1 - q : q;
    double2 t = tk[k], v = z[k];
    return 2.0 * (v.x * t.x + v.y * t.y);
  }
  int slot = (q & 1) ? n - 1 - (q >> 1) : (q >> 1);
  double y = z[slot].x;
  if (KIND == K_RODFT01 && (q & 1)) y = -y;
  return y;
}

// n = N1*N2 points per line; j = N2*j1 + j2, k = k1 + N1*k2:
//   Y[j2][k1] = sum_j1 z[N2 j1 + j2] W_N1^{j1 k1}, times W_n^{j2 k1}
//   Z[k1 + N1 k2] = sum_j2 Y[j2][k1] W_N2^{j2 k2}
// One task per thread in each pass (the host sizes L so that L*N1 and L*N2
// do not exceed the workgroup).  Y is stored row k1 with its N2 entries
// XOR-swizzled by k1, so both the pass-1 writes (consecutive j2) and the
// pass-2 reads (consecutive k1) spread over the LDS banks.  All IT loads of
// a thread are issued before its first LDS write.
template <int N1, int N2, int KIND, int LSHIFT>
__global__ __launch_bounds__(NT) void k_r2r_fft(Args a) {
  extern __shared__ double2 S[];
  constexpr int n = N1 * N2;
  constexpr int L = (fft_lines(N1, N2) >> LSHIFT) > 0 ? (fft_lines(N1, N2) >> LSHIFT) : 1;
  constexpr int IT = (L * n + NT - 1) / NT;  // elements per thread in the load / store phases
  const int line0 = blockIdx.x * L;
  const double2 *tw = reinterpret_cast<const double2 *>(a.tab);      // e^{-2 pi i m/n}, m < n
  const double2 *tk = reinterpret_cast<const double2 *>(a.tab) + n;  // (cos, sin)(pi k/2n)
  constexpr bool inv = (KIND == K_HC2R || KIND == K_REDFT01 || KIND == K_RODFT01);
  double *R = reinterpret_cast<double *>(S);
  __shared__ long oin[L], oout[L];
  line_offsets<L>(a, line0, oin, oout);
  // 1. raw lines into LDS, line l at doubles [2 n l, 2 n l + n)
  {
    double xr[IT];
#pragma unroll
    for (int it = 0; it < IT; it++) {
      const int e = threadIdx.x + it * NT;
      const int l = a.coal ? e % L : e / n, q = a.coal ? e / L : e % n;
      xr[it] = 0.0;
      if (e < L * n && oin[l] >= 0) xr[it] = a.in[q * a.ies + oin[l]];
    }
#pragma unroll
    for (int it = 0; it < IT; it++) {
      const int e = threadIdx.x + it * NT;
      const int l = a.coal ? e % L : e / n, q = a.coal ? e / L : e % n;
      if (e < L * n) R[2 * n * l + q] = xr[it];
    }
  }
  __syncthreads();
  // 2. first pass: N1-point DFTs over j1 for every (line, j2)
  {
    const int t = threadIdx.x;
    const bool act = t < L * N2;
    const int j2 = t % N2, l = t / N2;
    double2 v[N1];
    if (act) {
      const double *r = R + 2 * n * l;
#pragma unroll
      for (int j1 = 0; j1 < N1; j1++) v[j1] = pre_slot<KIND>(r, N2 * j1 + j2, n, tk);
      fft_reg<N1>(v, tw, N2, inv);
#pragma unroll
      for (int k1 = 1; k1 < N1; k1++) {
        double2 w = tw[(j2 * k1) & (n - 1)];
        if (inv) w.y = -w.y;
        double2 y = v[k1];
        v[k1] = make_double2(y.x * w.x - y.y * w.y, y.x * w.y + y.y * w.x);
      }
    }
    __syncthreads();
    if (act) {
      double2 *T = S + n * l;
#pragma unroll
      for (int k1 = 0; k1 < N1; k1++) T[k1 * N2 + (j2 ^ (k1 & (N2 - 1)))] = v[k1];
    }
    __syncthreads();
  }
  // 3. second pass: N2-point DFTs over j2 for every (line, k1)
  {
    const int t = threadIdx.x;
    const bool act = t < L * N1;
    const int k1 = t % N1, l = t / N1;
    double2 v[N2];
    if (act) {
      const double2 *T = S + n * l;
#pragma unroll
      for (int j2 = 0; j2 < N2; j2++) v[j2] = T[k1 * N2 + (j2 ^ (k1 & (N2 - 1)))];
      fft_reg<N2>(v, tw, N1, inv);
    }
    __syncthreads();
    if (act) {
      double2 *Z = S + n * l;
#pragma unroll
      for (int k2 = 0; k2 < N2; k2++) Z[k1 + N1 * k2] = v[k2];
    }
    __syncthreads();
  }
  // 4. post-mapping and store
#pragma unroll
  for (int it = 0; it < IT; it++) {
    const int e = threadIdx.x + it * NT;
    const int l = a.coal ? e % L : e / n, q = a.coal ? e / L : e % n;
    if (e < L * n && oout[l] >= 0) {
      const double y = post_val<KIND>(S + n * l, q, n, tk);
      a.out[q * a.oes + oout[l]] = y * a.scale;
    }
  }
}

// R2HC / HC2R of n = 2h points through one h-point complex FFT per line
// (h = N1*N2), half the work and half the LDS of the n-point form:
//   forward: z[m] = x[2m] + i x[2m+1]; Z = FFT_h(z); for k = 0..h
//     X[k] = E + W_n^k O,  E = (Z[k] + conj Z[h-k]) / 2,  O = (Z[k] - conj Z[h-k]) / 2i
//   inverse: Z[k] = A + i B,  A = X[k] + conj X[h-k],  B = (X[k] - conj X[h-k]) w^k
//     (w = e^{2 pi i/n}), z = IFFT_h(Z), y[2m] + i y[2m+1] = z[m]
// (indices of Z modulo h).  Every line is transformed on its own, so a line
// of zeros stays exactly zero.  The raw line and its h complex values share
// one n-double slot of LDS.
#ifndef SNAC_RFFT_PAD
#define SNAC_RFFT_PAD 2
#endif
constexpr int RPAD = SNAC_RFFT_PAD;  // doubles of padding after each LDS line (spreads lines over the banks)
constexpr int rfft_lines(int n1, int n2) {
  return (NT / (n1 > n2 ? n1 : n2)) < (LDS_COMPLEX / (2 * n1 * n2)) ? (NT / (n1 > n2 ? n1 : n2))
                                                                    : (LDS_COMPLEX / (2 * n1 * n2));
}

// The two passes of the h-point complex FFT of one line (h = N1*N2) and
// its unfolding.  The line's LDS slot holds the n = 2h raw doubles (r) and,
// after pass 1, its h complex values (T, XOR-swizzled between the passes,
// then Z in natural order).  k_rfft_w uses these; k_rfft keeps the same
// steps written inline, which the compiler allocates in fewer registers
// there (164 against 172 VGPRs for the n = 256 inverse: a wave per SIMD).
// Pass 1: N1-point DFT over j1 of column j2, the inverse's folding of the
// halfcomplex input on the way in, the twiddles W_h^{j2 k1} on the way out.
template <int N1, int N2, bool INV>
__device__ __forceinline__ void rfft_pass1(const double *r, int j2, const double2 *tw, double2 (&v)[N1]) {
  constexpr int h = N1 * N2, n = 2 * h;
#pragma unroll
  for (int j1 = 0; j1 < N1; j1++) {
    const int k = N2 * j1 + j2;
    if (!INV) {
      v[j1] = make_double2(r[2 * k], r[2 * k + 1]);
    } else {
      // X[k] and conj X[h-k] from the halfcomplex line
      const double2 xk = (k == 0) ? make_double2(r[0], 0.0) : make_double2(r[k], r[n - k]);
      const double2 xc = (k == 0) ? make_double2(r[h], 0.0) : make_double2(r[h - k], -r[h + k]);
      const double2 w = tw[k];  // conj of w^k
      const double dx = xk.x - xc.x, dy = xk.y - xc.y;
      const double bx = dx * w.x + dy * w.y, by = dy * w.x - dx * w.y;  // (dx + i dy) e^{+2 pi i k/n}
      v[j1] = make_double2(xk.x + xc.x - by, xk.y + xc.y + bx);        // A + i B
    }
  }
  fft_reg<N1>(v, tw, 2 * N2, INV);
#pragma unroll
  for (int k1 = 1; k1 < N1; k1++) {
    double2 w = tw[(2 * j2 * k1) & (n - 1)];
    if (INV) w.y = -w.y;
    const double2 y = v[k1];
    v[k1] = make_double2(y.x * w.x - y.y * w.y, y.x * w.y + y.y * w.x);
  }
}
template <int N1, int N2>
__device__ __forceinline__ void rfft_put1(double2 *T, int j2, const double2 (&v)[N1]) {
#pragma unroll
  for (int k1 = 0; k1 < N1; k1++) T[k1 * N2 + (j2 ^ (k1 & (N2 - 1)))] = v[k1];
}
// Pass 2: N2-point DFT over j2 of row k1
template <int N1, int N2, bool INV>
__device__ __forceinline__ void rfft_pass2(const double2 *T, int k1, const double2 *tw, double2 (&v)[N2]) {
#pragma unroll
  for (int j2 = 0; j2 < N2; j2++) v[j2] = T[k1 * N2 + (j2 ^ (k1 & (N2 - 1)))];
  fft_reg<N2>(v, tw, 2 * N1, INV);
}
template <int N1, int N2>
__device__ __forceinline__ void rfft_put2(double2 *Z, int k1, const double2 (&v)[N2]) {
#pragma unroll
  for (int k2 = 0; k2 < N2; k2++) Z[k1 + N1 * k2] = v[k2];
}
// Output q of the line from its h-point spectrum Z: forward, the halfcomplex
// X[q] (q <= h: real part, else the imaginary part of X[n-q]); inverse, the
// real sample y[q]
template <int N1, int N2, bool INV>
__device__ __forceinline__ double rfft_out(const double2 *Z, int q, const double2 *tw) {
  constexpr int h = N1 * N2, n = 2 * h;
  if (!INV) {
    const int k = q <= h ? q : n - q;
    const double2 zk = Z[k & (h - 1)], zc = Z[(h - k) & (h - 1)];  // Z[k], Z[h-k] (mod h)
    const double ex = 0.5 * (zk.x + zc.x), ey = 0.5 * (zk.y - zc.y);
    const double ox = 0.5 * (zk.y + zc.y), oy = -0.5 * (zk.x - zc.x);
    const double2 w = tw[k];
    const double xr = ex + (w.x * ox - w.y * oy), xi = ey + (w.x * oy + w.y * ox);
    return q <= h ? xr : xi;
  }
  const double2 z = Z[q >> 1];
  return (q & 1) ? z.y : z.x;
}

// TPB tiles of L lines per workgroup: the loads of tile t+1 are issued
// before tile t is transformed and land in LDS after it, so their latency
// overlaps the arithmetic (TPB = 1: one tile, no overlap).
template <int N1, int N2, bool INV, int LSHIFT, int TPB>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(N1 < N2 ? 4 : 1))) void k_rfft(Args a) {
  extern __shared__ double2 S[];
  constexpr int h = N1 * N2, n = 2 * h;
  constexpr int L = (rfft_lines(N1, N2) >> LSHIFT) > 0 ? (rfft_lines(N1, N2) >> LSHIFT) : 1;
  constexpr int IT = (L * n + NT - 1) / NT;
  const double2 *tw = reinterpret_cast<const double2 *>(a.tab);  // e^{-2 pi i m/n}, m < n
  constexpr int LS = n + RPAD;                                     // LDS doubles per line
  double *R = reinterpret_cast<double *>(S);                     // line l at doubles [LS l, LS l + n)
  __shared__ long oin[2][L], oout[2][L];
  const int ntile = (a.nlines + L - 1) / L, tile0 = blockIdx.x * TPB;
  auto offsets = [&](int slot, int tile) {
    for (int t = threadIdx.x; t < L; t += NT) {
      const int line = tile * L + t;
      long oi, oo;
      line_offset(a, line, oi, oo);
      oin[slot][t] = oi;
      oout[slot][t] = oo;
    }
  };
  double xr[IT];
  auto load = [&](int slot) {
#pragma unroll
    for (int it = 0; it < IT; it++) {
      const int e = threadIdx.x + it * NT;
      const int l = a.coal ? e % L : e / n, q = a.coal ? e / L : e % n;
      xr[it] = 0.0;
      if (e < L * n && oin[slot][l] >= 0) xr[it] = a.in[q * a.ies + oin[slot][l]];
    }
  };
  offsets(0, tile0);
  __syncthreads();
  load(0);
  for (int tt = 0; tt < TPB; tt++) {
  const int tile = tile0 + tt;
  if (tile >= ntile) break;  // uniform over the workgroup
  const int sl = tt & 1;
  const bool more = tt + 1 < TPB && tile + 1 < ntile;
  __syncthreads();  // the previous tile is done with the LDS lines and its offsets
  // 1. raw lines into LDS
#pragma unroll
  for (int it = 0; it < IT; it++) {
    const int e = threadIdx.x + it * NT;
    const int l = a.coal ? e % L : e / n, q = a.coal ? e / L : e % n;
    if (e < L * n) R[LS * l + q] = xr[it];
  }
  if (more) offsets(sl ^ 1, tile + 1);
  __syncthreads();
  if (more) load(sl ^ 1);
  // 2. first pass: N1-point DFTs over j1 for every (line, j2)
  {
    const int t = threadIdx.x;
    const bool act = t < L * N2;
    const int j2 = t % N2, l = t / N2;
    double2 v[N1];
    if (act) {
      const double *r = R + LS * l;
#pragma unroll
      for (int j1 = 0; j1 < N1; j1++) {
        const int k = N2 * j1 + j2;
        if (!INV) {
          v[j1] = make_double2(r[2 * k], r[2 * k + 1]);
        } else {
          // X[k] and conj X[h-k] from the halfcomplex line
          const double2 xk = (k == 0) ? make_double2(r[0], 0.0) : make_double2(r[k], r[n - k]);
          const double2 xc = (k == 0) ? make_double2(r[h], 0.0) : make_double2(r[h - k], -r[h + k]);
          const double2 w = tw[k];  // conj of w^k
          const double dx = xk.x - xc.x, dy = xk.y - xc.y;
          const double bx = dx * w.x + dy * w.y, by = dy * w.x - dx * w.y;  // (dx + i dy) e^{+2 pi i k/n}
          v[j1] = make_double2(xk.x + xc.x - by, xk.y + xc.y + bx);        // A + i B
        }
      }
      fft_any<N1>(v, tw, 2 * N2, INV);
#pragma unroll
      for (int k1 = 1; k1 < N1; k1++) {
        double2 w = tw[2 * j2 * k1];  // 2 j2 k1 < n
        if (INV) w.y = -w.y;
        double2 y = v[k1];
        v[k1] = make_double2(y.x * w.x - y.y * w.y, y.x * w.y + y.y * w.x);
      }
    }
    __syncthreads();
    if (act) {
      double2 *T = S + (LS / 2) * l;
#pragma unroll
      for (int k1 = 0; k1 < N1; k1++) T[k1 * N2 + (j2 ^ (k1 & (N2 - 1)))] = v[k1];
    }
    __syncthreads();
  }
  // 3. second pass: N2-point DFTs over j2 for every (line, k1)
  {
    const int t = threadIdx.x;
    const bool act = t < L * N1;
    const int k1 = t % N1, l = t / N1;
    double2 v[N2];
    if (act) {
      const double2 *T = S + (LS / 2) * l;
#pragma unroll
      for (int j2 = 0; j2 < N2; j2++) v[j2] = T[k1 * N2 + (j2 ^ (k1 & (N2 - 1)))];
      fft_reg<N2>(v, tw, 2 * N1, INV);
    }
    __syncthreads();
    if (act) {
      double2 *Z = S + (LS / 2) * l;
#pragma unroll
      for (int k2 = 0; k2 < N2; k2++) Z[k1 + N1 * k2] = v[k2];
    }
    __syncthreads();
  }
  // 4. post-mapping and store
#pragma unroll
  for (int it = 0; it < IT; it++) {
    const int e = threadIdx.x + it * NT;
    const int l = a.coal ? e % L : e / n, q = a.coal ? e / L : e % n;
    if (e < L * n && oout[sl][l] >= 0) {
      const double2 *Z = S + (LS / 2) * l;
      double y;
      if (!INV) {
        const int k = q <= h ? q : n - q;
        const double2 zk = Z[k < h ? k : 0], zc = Z[k > 0 ? h - k : 0];  // Z[k], Z[h-k] (mod h)
        const double ex = 0.5 * (zk.x + zc.x), ey = 0.5 * (zk.y - zc.y);
        const double ox = 0.5 * (zk.y + zc.y), oy = -0.5 * (zk.x - zc.x);
        const double2 w = tw[k];
        const double xr = ex + (w.x * ox - w.y * oy), xi = ey + (w.x * oy + w.y * ox);
        y = q <= h ? xr : xi;
      } else {
        const double2 z = Z[q >> 1];
        y = (q & 1) ? z.y : z.x;
      }
      a.out[q * a.oes + oout[sl][l]] = y * a.scale;
    }
  }
  }
}

// Orders this wavefront's LDS accesses before and after it: a wavefront's
// LDS instructions execute in issue order, so lanes of one wavefront see each
// other's writes without a workgroup barrier once the compiler keeps the
// order (the fences at wavefront scope and the scheduling barrier).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The same transform with each wavefront owning LW = L/4 of the workgroup's
// L lines through both passes, so the passes need no workgroup barrier.
// Contiguous lines (stride 1) are also loaded and stored by their own
// wavefront (one barrier in all, for the line offsets); strided lines are
// loaded and stored by the whole workgroup, 8L contiguous bytes per row,
// with a barrier after the load and one before the store.  Compiled for
// four waves per SIMD (at most 128 VGPRs, a few spilled), which measured
// faster than three without spills.
template <int N1, int N2, bool INV>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_rfft_w(Args a) {
  extern __shared__ double2 S[];
  constexpr int h = N1 * N2, n = 2 * h;
  constexpr int L = rfft_lines(N1, N2), LW = L / 4;
  static_assert(NT == 256 && L % 4 == 0 && LW * N1 <= 64 && LW * N2 <= 64 && (L * n) % NT == 0,
                "one pass task per lane of the owning wavefront");
  constexpr int IT = L * n / NT;  // = LW * n / 64
  const double2 *tw = reinterpret_cast<const double2 *>(a.tab);
  constexpr int LS = n + RPAD;
  double *R = reinterpret_cast<double *>(S);
  __shared__ long oin[L], oout[L];
  const int wv = threadIdx.x >> 6, ln = threadIdx.x & 63;
  for (int t = threadIdx.x; t < L; t += NT) {
    const int line = blockIdx.x * L + t;
    long oi, oo;
    line_offset(a, line, oi, oo);
    oin[t] = oi;
    oout[t] = oo;
  }
  __syncthreads();
  const bool coal = a.coal;
  // element it of this thread: line l, position q
  auto elem = [&](int it, int &l, int &q) {
    if (coal) {
      const int e = threadIdx.x + it * NT;
      l = e % L;
      q = e / L;
    } else {
      const int e = ln + it * 64;
      l = wv * LW + e / n;
      q = e % n;
    }
  };
  // 1. raw lines into LDS
  {
    double xr[IT];
#pragma unroll
    for (int it = 0; it < IT; it++) {
      int l, q;
      elem(it, l, q);
      xr[it] = oin[l] >= 0 ? a.in[q * a.ies + oin[l]] : 0.0;
    }
#pragma unroll
    for (int it = 0; it < IT; it++) {
      int l, q;
      elem(it, l, q);
      R[LS * l + q] = xr[it];
    }
  }
  if (coal) __syncthreads();
  else wave_sync();
  // 2. first pass over this wavefront's lines
  {
    const bool act = ln < LW * N2;
    const int j2 = ln % N2, l = wv * LW + ln / N2;
    double2 v[N1];
    if (act) rfft_pass1<N1, N2, INV>(R + LS * l, j2, tw, v);
    wave_sync();
    if (act) rfft_put1<N1, N2>(S + (LS / 2) * l, j2, v);
    wave_sync();
  }
  // 3. second pass
  {
    const bool act = ln < LW * N1;
    const int k1 = ln % N1, l = wv * LW + ln / N1;
    double2 v[N2];
    if (act) rfft_pass2<N1, N2, INV>(S + (LS / 2) * l, k1, tw, v);
    wave_sync();
    if (act) rfft_put2<N1, N2>(S + (LS / 2) * l, k1, v);
    wave_sync();
  }
  if (coal) __syncthreads();
  // 4. post-mapping and store
#pragma unroll
  for (int it = 0; it < IT; it++) {
    int l, q;
    elem(it, l, q);
    if (oout[l] >= 0) a.out[q * a.oes + oout[l]] = rfft_out<N1, N2, INV>(S + (LS / 2) * l, q, tw) * a.scale;
  }
}

// Dense transforms on the FP64 matrix cores: the kinds and lengths without a
// power-of-two FFT.  A transform of n points is a matrix product Y = M X over
// the lines; most kinds' matrices are symmetric or antisymmetric under a
// mirror of the samples (j -> n - j for R2HC / HC2R, n - 1 - j for the cosine
// and sine kinds), so the product splits into a symmetric and an
// antisymmetric part of half the size each, half the multiplications:
//   MODE 1 (R2HC, REDFT10, RODFT10, RODFT00): the input is folded,
//     s_j = x_j + x_mirror, a_j = x_j - x_mirror as it is loaded;
//   MODE 2 (HC2R, REDFT01, RODFT01): the output is unfolded,
//     y_j = E_j + O_j, y_mirror = E_j - O_j;
//   MODE 0 (REDFT11, RODFT11): no fold.
// A workgroup holds L = 16 NTL LG lines in LDS; each of its wavefronts takes
// tiles of 16 matrix rows for 16 NTL of them (v_mfma_f64_16x16x4).  The
// matrix comes from memory in the instruction's operand order, 512
// contiguous bytes per load, L2-resident and used for NTL products.  With
// SWAP (outputs contiguous along the line) the operands change places, so
// that the 16 lanes of a result row hold consecutive outputs of one line and
// the stores are 128-byte runs either way.
// Bound: 2 n (MODE 0) or n FP64 operations per point at the matrix rate (72
// TFLOP/s measured on a large product) against 16 bytes per point; at n = 192
// the folded product takes about as long as the memory does.  The form it
// replaces walked a matrix row per thread (8-byte loads a row apart): 347 us
// on average over the transforms of a 192x96x96 box, 16-26 us this way; 146 ->
// 12-18 us for a 180x77x90 channel's (0.8 TB/s of the lines' bytes), 8.1 ->
// 3.4 us for two-point lines.
typedef double double4_ __attribute__((ext_vector_type(4)));
struct MJob {  // one batch of lines and its first workgroup
  const double *in;
  double *out;
  long ies, is1, is2, oes, os1, os2;
  int nb1, nlines, start;
};
struct MArgs {
  MJob job[GRID_BLOCKS];
  int njob;
  const double *fs, *fa;  // matrix fragments [tile][k / 4][64] of the two parts
  double scale;
  int n;
  int half;     // samples up to the mirror (MODE 0: n)
  int rows;     // matrix rows of the symmetric part (MODE 2: of both)
  int ks, ka;   // inner lengths of the two parts
  int na;       // MODE 1: rows of the antisymmetric part
  int hc;       // 1: R2HC / HC2R index maps, 0: even / odd
  int ld, ntile, tw, lg;
};

template <int MODE, bool SWAP, int NTL>
__global__ __launch_bounds__(512) void k_r2r_mfma(MArgs a) {
  extern __shared__ double2 S[];
  const int L = 16 * NTL * a.lg, nthr = 64 * a.tw * a.lg, n = a.n;
  double *X = reinterpret_cast<double *>(S);  // [L][ld]: symmetric part, then (at ksp) the antisymmetric one
  long *oin = reinterpret_cast<long *>(X + (size_t)L * a.ld), *oout = oin + L;
  const int ksp = (a.ks + 3) & ~3, kap = (a.ka + 3) & ~3;
  int q = 0;
  while (q + 1 < a.njob && (int)blockIdx.x >= a.job[q + 1].start) q++;
  const MJob &J = a.job[q];
  const int line0 = (blockIdx.x - J.start) * L;
  for (int t = threadIdx.x; t < L; t += nthr) {
    const int line = line0 + t;
    long oi = -1, oo = -1;
    if (line < J.nlines) {
      const int b1 = line % J.nb1, b2 = line / J.nb1;
      oi = b1 * J.is1 + b2 * J.is2;
      oo = b1 * J.os1 + b2 * J.os2;
    }
    oin[t] = oi;
    oout[t] = oo;
  }
  __syncthreads();
  // 1. lines into LDS: folded (MODE 1), sorted into the two parts (MODE 2) or
  // as they are; the inner dimension's padding is zero
  const int cols = MODE == 1 ? a.half : n;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ln = threadIdx.x & 63;
  constexpr int U = 4;  // elements (MODE 1: pairs) in flight per thread
  auto mirror = [&](int j) { return a.hc ? (j == 0 ? 0 : n - j) : n - 1 - j; };
  auto put = [&](double *row, int j, double x, double y) {
    if (MODE == 1) {
      row[j] = x + y;
      if (j < a.ka) row[ksp + j] = mirror(j) != j ? x - y : 0.0;
    } else if (MODE == 2) {
      if (a.hc) row[j < a.ks ? j : ksp + n - 1 - j] = x;
      else row[(j & 1) ? ksp + (j >> 1) : j >> 1] = x;
    } else {
      row[j] = x;
    }
  };
  if (J.ies != 1) {  // strided lines: consecutive threads on consecutive lines, one line per thread
    const int lsh = __ffs(L) - 1, l = threadIdx.x & (L - 1), js = nthr >> lsh;  // L is a power of two dividing nthr
    const long o = oin[l];
    double *row = X + l * a.ld;
    const double *p = J.in + (o >= 0 ? o : 0);
    for (int j0 = threadIdx.x >> lsh; j0 < cols; j0 += js * U) {
      double x[U], y[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int j = j0 + u * js;
        const bool ok = o >= 0 && j < cols;
        x[u] = ok ? p[j * J.ies] : 0.0;
        y[u] = MODE == 1 && ok && mirror(j) != j ? p[mirror(j) * J.ies] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < U; u++)
        if (j0 + u * js < cols) put(row, j0 + u * js, x[u], y[u]);
    }
  } else if (cols < 48) {  // short contiguous lines: samples of several lines per wavefront
    for (int e0 = threadIdx.x; e0 < L * cols; e0 += nthr * U) {
      double x[U], y[U];
      int l[U], j[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int e = e0 + u * nthr;
        l[u] = min(e / cols, L - 1);
        j[u] = e - l[u] * cols;
        const long o = oin[l[u]];
        const bool ok = o >= 0 && j[u] < cols;
        const double *p = J.in + o;
        x[u] = ok ? p[j[u]] : 0.0;
        y[u] = MODE == 1 && ok && mirror(j[u]) != j[u] ? p[mirror(j[u])] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < U; u++)
        if (j[u] < cols) put(X + l[u] * a.ld, j[u], x[u], y[u]);
    }
  } else {  // contiguous lines: a wavefront on 64 samples of a line
    const int nch = (cols + 63) >> 6, nw = a.tw * a.lg, tot = (L / nw + (wv < L % nw ? 1 : 0)) * nch;
    for (int t0 = 0; t0 < tot; t0 += U) {
      double x[U], y[U];
      int l[U], j[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int t = t0 + u, q = t / nch;
        l[u] = min(wv + q * nw, L - 1);
        j[u] = t < tot ? ((t - q * nch) << 6) + ln : cols;
        const long o = oin[l[u]];
        const bool ok = o >= 0 && j[u] < cols;
        const double *p = J.in + o;
        x[u] = ok ? p[j[u]] : 0.0;
        y[u] = MODE == 1 && ok && mirror(j[u]) != j[u] ? p[mirror(j[u])] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < U; u++)
        if (j[u] < cols) put(X + l[u] * a.ld, j[u], x[u], y[u]);
    }
  }
  for (int l = threadIdx.x; l < L; l += nthr) {
    double *row = X + l * a.ld;
    for (int k = a.ks; k < ksp; k++) row[k] = 0.0;
    for (int k = a.ka; k < kap; k++) row[ksp + k] = 0.0;
  }
  __syncthreads();
  const int lq = ln & 15, kq = ln >> 4, l0 = (wv / a.tw) * 16 * NTL;
  for (int tile = wv % a.tw; tile < a.ntile; tile += a.tw) {
    double4_ es[NTL], ea[NTL];
#pragma unroll
    for (int t = 0; t < NTL; t++) { es[t] = double4_{0, 0, 0, 0}; ea[t] = double4_{0, 0, 0, 0}; }
    // 2. the two products; operand layout: lane -> (row or column ln & 15, inner ln >> 4)
    const double *xs = X + (l0 + lq) * a.ld + kq;
    auto step = [&](double m, const double *x, int k, double4_ (&acc)[NTL]) {
#pragma unroll
      for (int t = 0; t < NTL; t++) {
        const double b = x[t * 16 * a.ld + 4 * k];
        acc[t] = SWAP ? __builtin_amdgcn_mfma_f64_16x16x4f64(b, m, acc[t], 0, 0, 0)
                      : __builtin_amdgcn_mfma_f64_16x16x4f64(m, b, acc[t], 0, 0, 0);
      }
    };
    // both parts side by side, the matrix values of the next W inner blocks
    // loaded before this one's products (W of either part in flight)
    constexpr int W = 4;
    const int nks = ksp / 4, nka = MODE != 0 ? kap / 4 : 0;
    const double *fs = a.fs + (size_t)tile * nks * 64 + ln, *fa = a.fa + (size_t)tile * nka * 64 + ln;
    const int nk = MODE != 0 ? min(nks, nka) : nks, nw = nk / W * W;
    double ms[W], ma[W];
    if (nw > 0) {
#pragma unroll
      for (int u = 0; u < W; u++) {
        ms[u] = fs[u * 64];
        if (MODE != 0) ma[u] = fa[u * 64];
      }
    }
    for (int k = 0; k < nw; k += W) {
      double ns[W], na[W];
      const bool more = k + W < nw;
#pragma unroll
      for (int u = 0; u < W; u++) {
        ns[u] = more ? fs[(size_t)(k + W + u) * 64] : 0.0;
        if (MODE != 0) na[u] = more ? fa[(size_t)(k + W + u) * 64] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < W; u++) {
        step(ms[u], xs, k + u, es);
        if (MODE != 0) step(ma[u], xs + ksp, k + u, ea);
      }
#pragma unroll
      for (int u = 0; u < W; u++) {
        ms[u] = ns[u];
        if (MODE != 0) ma[u] = na[u];
      }
    }
    for (int k = nw; k < nks; k++) step(fs[(size_t)k * 64], xs, k, es);
    for (int k = nw; k < nka; k++) step(fa[(size_t)k * 64], xs + ksp, k, ea);
    // 3. results: register v of a lane is row 4 v + (ln >> 4), column ln & 15
    const long oes = SWAP ? 1 : J.oes;
#pragma unroll
    for (int t = 0; t < NTL; t++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int l = l0 + 16 * t + (SWAP ? 4 * v + kq : lq), r = 16 * tile + (SWAP ? lq : 4 * v + kq);
        const long o = oout[l];
        if (o < 0 || r >= a.rows) continue;
        double *y = J.out + o;
        if (MODE == 0) {
          y[r * oes] = es[t][v] * a.scale;
        } else if (MODE == 1) {
          y[(a.hc ? r : 2 * r) * oes] = es[t][v] * a.scale;
          if (r < a.na) y[(a.hc ? n - 1 - r : 2 * r + 1) * oes] = ea[t][v] * a.scale;
        } else {
          const int mir = mirror(r);
          y[r * oes] = (es[t][v] + ea[t][v]) * a.scale;
          if (mir != r) y[mir * oes] = (es[t][v] - ea[t][v]) * a.scale;
        }
      }
  }
}

// The dense product one output per thread: lengths past the matrix-core
// form's LDS, and the mixed-precision mode's transforms.  There FP32
// right-hand sides turn any change of rounding, however small, into
// differences of about 2e-9 of the velocities within a few substages (its own
// error is 6.6e-8).  That mode was left with its operations, their order and
// the coefficients of r2r_coef so that its results stay what they were, not for
// their accuracy.
__global__ __launch_bounds__(NT) void k_r2r_dense(Args a) {
  extern __shared__ double2 S[];
  double *R = reinterpret_cast<double *>(S);
  const int n = a.n, L = a.L, line0 = blockIdx.x * L;
  for (int e = threadIdx.x; e < L * n; e += NT) {
    int l, q;
    elem_of(a, e, l, q);
    int line = line0 + l;
    if (line >= a.nlines) continue;
    int b1 = line % a.nb1, b2 = line / a.nb1;
    R[l * n + q] = a.in[q * a.ies + b1 * a.is1 + b2 * a.is2];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < L * n; e += NT) {
    int l, q;
    elem_of(a, e, l, q);
    int line = line0 + l;
    if (line >= a.nlines) continue;
    const double *row = a.tab + (long)q * n;
    const double *x = R + l * n;
    double y = 0.0;
    for (int j = 0; j < n; j++) y += row[j] * x[j];
    int b1 = line % a.nb1, b2 = line / a.nb1;
    a.out[q * a.oes + b1 * a.os1 + b2 * a.os2] = y * a.scale;
  }
}

// n = N1 * N2 with both factors as even as possible
void fft_split(int n, int &n1, int &n2) {
  int lg = 0;
  while ((1 << lg) < n) lg++;
  n2 = 1 << (lg / 2);
  n1 = n / n2;
}

template <int N1, int N2, int LS>
void launch_sized_l(int kind, dim3 grid, size_t lds, hipStream_t s, const Args &a) {
  switch (kind) {
  case K_R2HC: hipLaunchKernelGGL((k_r2r_fft<N1, N2, K_R2HC, LS>), grid, dim3(NT), lds, s, a); break;
  case K_HC2R: hipLaunchKernelGGL((k_r2r_fft<N1, N2, K_HC2R, LS>), grid, dim3(NT), lds, s, a); break;
  case K_REDFT10: hipLaunchKernelGGL((k_r2r_fft<N1, N2, K_REDFT10, LS>), grid, dim3(NT), lds, s, a); break;
  case K_REDFT01: hipLaunchKernelGGL((k_r2r_fft<N1, N2, K_REDFT01, LS>), grid, dim3(NT), lds, s, a); break;
  case K_RODFT10: hipLaunchKernelGGL((k_r2r_fft<N1, N2, K_RODFT10, LS>), grid, dim3(NT), lds, s, a); break;
  case K_RODFT01: hipLaunchKernelGGL((k_r2r_fft<N1, N2, K_RODFT01, LS>), grid, dim3(NT), lds, s, a); break;
  default: throw std::runtime_error("r2r: kind has no FFT path");
  }
}

template <int N1, int N2>
void launch_sized(int kind, int lshift, dim3 grid, size_t lds, hipStream_t s, const Args &a) {
  switch (lshift) {
  case 0: launch_sized_l<N1, N2, 0>(kind, grid, lds, s, a); break;
  case 1: launch_sized_l<N1, N2, 1>(kind, grid, lds, s, a); break;
  case 2: launch_sized_l<N1, N2, 2>(kind, grid, lds, s, a); break;
  default: throw std::runtime_error("r2r: bad tile choice");
  }
}

void launch_fft_kind(int kind, int n, int ls, dim3 grid, size_t lds, hipStream_t s, const Args &a) {
  switch (n) {
  case 4: launch_sized<2, 2>(kind, ls, grid, lds, s, a); break;
  case 8: launch_sized<4, 2>(kind, ls, grid, lds, s, a); break;
  case 16: launch_sized<4, 4>(kind, ls, grid, lds, s, a); break;
  case 32: launch_sized<8, 4>(kind, ls, grid, lds, s, a); break;
  case 64: launch_sized<8, 8>(kind, ls, grid, lds, s, a); break;
  case 128: launch_sized<16, 8>(kind, ls, grid, lds, s, a); break;
  case 256: launch_sized<16, 16>(kind, ls, grid, lds, s, a); break;
  case 512: launch_sized<32, 16>(kind, ls, grid, lds, s, a); break;
  case 1024: launch_sized<32, 32>(kind, ls, grid, lds, s, a); break;
  default: throw std::runtime_error("r2r: no FFT path for length " + std::to_string(n));
  }
}

// tile 0..2: 2^-tile of the lines per workgroup; 3 / 4: full tiles, 2 / 4 per workgroup;
// 5: full tiles, wavefront-local passes (k_rfft_w); 6: full tiles, swapped split;
// 7: wavefront-local passes, swapped split
int rfft_tpb(int tile) { return tile == 3 ? 2 : (tile == 4 ? 4 : 1); }

template <int N1, int N2>
void launch_rfft_sized(bool inv, int tile, dim3 grid, size_t lds, hipStream_t s, const Args &a) {
#define SNAC_RF(I, LS, T) hipLaunchKernelGGL((k_rfft<N1, N2, I, LS, T>), grid, dim3(NT), lds, s, a)
  if (tile == 0) { if (inv) SNAC_RF(true, 0, 1); else SNAC_RF(false, 0, 1); }
  else if (tile == 1) { if (inv) SNAC_RF(true, 1, 1); else SNAC_RF(false, 1, 1); }
  else if (tile == 2) { if (inv) SNAC_RF(true, 2, 1); else SNAC_RF(false, 2, 1); }
  else if (tile == 3) { if (inv) SNAC_RF(true, 0, 2); else SNAC_RF(false, 0, 2); }
  else if (tile == 4) { if (inv) SNAC_RF(true, 0, 4); else SNAC_RF(false, 0, 4); }
  else if (tile == 5) {
    if (inv) hipLaunchKernelGGL((k_rfft_w<N1, N2, true>), grid, dim3(NT), lds, s, a);
    else hipLaunchKernelGGL((k_rfft_w<N1, N2, false>), grid, dim3(NT), lds, s, a);
  }
  else throw std::runtime_error("r2r: bad tile choice");
#undef SNAC_RF
}

// tiles 6 / 7: full tiles (7: wavefront-local passes) with the h-point FFT
// split the other way round (the shorter pass first, over all of a tile's
// threads)
template <int N1, int N2>
void launch_rfft_swapped(bool inv, bool wave, dim3 grid, size_t lds, hipStream_t s, const Args &a) {
  if (wave) {
    if (inv) hipLaunchKernelGGL((k_rfft_w<N1, N2, true>), grid, dim3(NT), lds, s, a);
    else hipLaunchKernelGGL((k_rfft_w<N1, N2, false>), grid, dim3(NT), lds, s, a);
  } else {
    if (inv) hipLaunchKernelGGL((k_rfft<N1, N2, true, 0, 1>), grid, dim3(NT), lds, s, a);
    else hipLaunchKernelGGL((k_rfft<N1, N2, false, 0, 1>), grid, dim3(NT), lds, s, a);
  }
}

// Mixed-radix lengths n = 2 N1 N2 (N1 with factors 3 and 5, N2 a power of two):
// the same kernel; the split of each length, or false.  From n = 72 on: there
// the matrix product's 2 n^2 operations a line take longer than its memory
// traffic (a 192x96x96 box: 96-point lines 16 -> 12-14 us, 192-point lines
// 23-26 -> 12-15 us); at 48 points both take 8 us, and the product takes
// several grid blocks in one launch.  These twelve lengths have instances and
// no others: the remaining even lengths with factors 2, 3 and 5 would gain as
// well, the more the longer, and take the product for now (64 x 64 lines of 180
// points 12-13 us, 360 25-27, 576 50-57, 960 126-128; of 384 points here 13-15).
bool rfft_mixed_split(int n, int &n1, int &n2) {
  static const int t[][3] = {{72, 9, 4},   {80, 5, 8},   {96, 6, 8},    {120, 15, 4},  {144, 9, 8},  {160, 10, 8},
                             {192, 12, 8}, {240, 15, 8}, {288, 9, 16}, {320, 10, 16}, {384, 12, 16}, {480, 15, 16}};
  for (auto &e : t)
    if (e[0] == n) {
      n1 = e[1];
      n2 = e[2];
      return true;
    }
  return false;
}
template <int N1, int N2>
void launch_rfft_mixed_sized(bool inv, int ls, dim3 grid, size_t lds, hipStream_t s, const Args &a) {
  if (ls == 0) {
    if (inv) hipLaunchKernelGGL((k_rfft<N1, N2, true, 0, 1>), grid, dim3(NT), lds, s, a);
    else hipLaunchKernelGGL((k_rfft<N1, N2, false, 0, 1>), grid, dim3(NT), lds, s, a);
  } else {
    if (inv) hipLaunchKernelGGL((k_rfft<N1, N2, true, 1, 1>), grid, dim3(NT), lds, s, a);
    else hipLaunchKernelGGL((k_rfft<N1, N2, false, 1, 1>), grid, dim3(NT), lds, s, a);
  }
}
void launch_rfft_mixed(bool inv, int n, int ls, dim3 grid, size_t lds, hipStream_t s, const Args &a) {
#define SNAC_MX(N, A, B) case N: launch_rfft_mixed_sized<A, B>(inv, ls, grid, lds, s, a); break;
  switch (n) {
    SNAC_MX(72, 9, 4) SNAC_MX(80, 5, 8)
    SNAC_MX(96, 6, 8) SNAC_MX(120, 15, 4) SNAC_MX(144, 9, 8) SNAC_MX(160, 10, 8) SNAC_MX(192, 12, 8)
    SNAC_MX(240, 15, 8) SNAC_MX(288, 9, 16) SNAC_MX(320, 10, 16) SNAC_MX(384, 12, 16) SNAC_MX(480, 15, 16)
    default: throw std::runtime_error("r2r: no mixed-radix path for length " + std::to_string(n));
  }
#undef SNAC_MX
}

// h-point split of an n = 2h point real transform
void launch_rfft(bool inv, int n, int ls, dim3 grid, size_t lds, hipStream_t s, const Args &a) {
  const bool sw = ls == 6 || ls == 7, wv = ls == 7;
  switch (n) {
  case 8: launch_rfft_sized<2, 2>(inv, sw ? (wv ? 5 : 0) : ls, grid, lds, s, a); break;
  case 16:
    if (sw) launch_rfft_swapped<2, 4>(inv, wv, grid, lds, s, a);
    else launch_rfft_sized<4, 2>(inv, ls, grid, lds, s, a);
    break;
  case 32: launch_rfft_sized<4, 4>(inv, sw ? (wv ? 5 : 0) : ls, grid, lds, s, a); break;
  case 64:
    if (sw) launch_rfft_swapped<4, 8>(inv, wv, grid, lds, s, a);
    else launch_rfft_sized<8, 4>(inv, ls, grid, lds, s, a);
    break;
  case 128: launch_rfft_sized<8, 8>(inv, sw ? (wv ? 5 : 0) : ls, grid, lds, s, a); break;
  case 256:
    if (sw) launch_rfft_swapped<8, 16>(inv, wv, grid, lds, s, a);
    else launch_rfft_sized<16, 8>(inv, ls, grid, lds, s, a);
    break;
  case 512: launch_rfft_sized<16, 16>(inv, sw ? (wv ? 5 : 0) : ls, grid, lds, s, a); break;
  case 1024:
    if (sw) launch_rfft_swapped<16, 32>(inv, wv, grid, lds, s, a);
    else launch_rfft_sized<32, 16>(inv, ls, grid, lds, s, a);
    break;
  default: throw std::runtime_error("r2r: no real-FFT path for length " + std::to_string(n));
  }
}

// ---- the matrix-core form: index maps, fragments, launch shape ----
// the split of kind's matrix under the mirror (k_r2r_mfma); Y[r] of a part is
// the sum over c of coef(out(r), in(c))
struct MSplit {
  int mode, hc, half, rows, na, ks, ka;
};
MSplit mfma_split(int kind, int n) {
  MSplit m{};
  m.hc = kind == K_R2HC || kind == K_HC2R;
  m.mode = kind == K_REDFT11 || kind == K_RODFT11                                                 ? 0
           : kind == K_HC2R || kind == K_REDFT01 || kind == K_RODFT01                             ? 2
                                                                                                  : 1;
  if (m.mode == 0) {
    m.half = m.rows = m.ks = n;
    return m;
  }
  m.half = m.hc ? n / 2 + 1 : (n + 1) / 2;
  const int sym = m.half, anti = n - m.half;  // the sizes of the two parts on the transformed side
  if (m.mode == 1) {
    m.rows = sym;
    m.na = anti;
    m.ks = m.ka = m.half;
  } else {
    m.rows = m.half;
    m.ks = sym;
    m.ka = anti;
  }
  return m;
}

// LDS doubles per line: both parts, padded to a row that is an odd multiple
// of two doubles, so that the 16 lines of an operand read fall on different banks
int mfma_ld(const MSplit &m) {
  const int ld = ((m.ks + 3) & ~3) + ((m.ka + 3) & ~3);
  return ld + 2;  // a multiple of 4, plus 2
}
size_t mfma_lds(int ld, int lines) { return (size_t)lines * (ld * sizeof(double) + 2 * sizeof(long)); }
constexpr size_t LDS_MAX = 160 * 1024;
// whether 16 lines fit (n up to about 1270; longer lines keep k_r2r_dense)
bool mfma_fits(int kind, int n) { return mfma_lds(mfma_ld(mfma_split(kind, n)), 16) <= LDS_MAX; }

// cos and sin of pi p / q, the angle reduced in integers first: p reaches n^2,
// and rounding the full-size angle would cost n ulps of the coefficient
double cos_pi(long p, long q) { return std::cos(std::acos(-1.0) * (double)(p % (2 * q)) / (double)q); }
double sin_pi(long p, long q) { return std::sin(std::acos(-1.0) * (double)(p % (2 * q)) / (double)q); }

double reduced_coef(int kind, int n_, int k_, int j_) {
  const long n = n_, k = k_, j = j_;
  switch (kind) {
  case K_R2HC:
    if (k <= n / 2) return cos_pi(2 * j * k, n);
    return -sin_pi(2 * j * (n - k), n);
  case K_HC2R:
    if (j == 0) return 1.0;
    if (n % 2 == 0 && j == n / 2) return (k % 2) ? -1.0 : 1.0;
    if (j < (n + 1) / 2) return 2.0 * cos_pi(2 * j * k, n);
    return -2.0 * sin_pi(2 * (n - j) * k, n);
  case K_REDFT10: return 2.0 * cos_pi((2 * j + 1) * k, 2 * n);
  case K_REDFT01: return j == 0 ? 1.0 : 2.0 * cos_pi(j * (2 * k + 1), 2 * n);
  case K_RODFT10: return 2.0 * sin_pi((2 * j + 1) * (k + 1), 2 * n);
  case K_RODFT01: return j == n - 1 ? ((k % 2) ? -1.0 : 1.0) : 2.0 * sin_pi((j + 1) * (2 * k + 1), 2 * n);
  case K_REDFT11: return 2.0 * cos_pi((2 * j + 1) * (2 * k + 1), 4 * n);
  case K_RODFT11: return 2.0 * sin_pi((2 * j + 1) * (2 * k + 1), 4 * n);
  // DST-I: the transform of a staggered Dirichlet-Dirichlet axis (fft.f90:130-133)
  case K_RODFT00: return 2.0 * sin_pi((j + 1) * (k + 1), n + 1);
  default: throw std::runtime_error("unsupported r2r kind " + std::to_string(kind));
  }
}

std::vector<double> mfma_fragments(int kind, int n) {
  const MSplit m = mfma_split(kind, n);
  const int nt = (m.rows + 15) / 16, kb[2] = {(m.ks + 3) / 4, (m.ka + 3) / 4};
  std::vector<double> f((size_t)nt * 64 * (kb[0] + kb[1]), 0.0);
  for (int part = 0; part < 2; part++) {
    const int nr = part == 0 ? m.rows : (m.mode == 1 ? m.na : m.rows), nc = part == 0 ? m.ks : m.ka;
    auto side = [&](int q) { return m.hc ? (part == 0 ? q : n - 1 - q) : 2 * q + part; };  // transformed side
    double *out = f.data() + (part == 0 ? 0 : (size_t)nt * kb[0] * 64);
    for (int r = 0; r < nr; r++)
      for (int c = 0; c < nc; c++) {
        // the antisymmetric part has nothing on a sample that is its own mirror
        const int sample = m.mode == 1 ? c : r;
        if (m.mode != 0 && part == 1 && sample == (m.hc ? (n - sample) % n : n - 1 - sample)) continue;
        const double v = m.mode == 0   ? reduced_coef(kind, n, r, c)
                         : m.mode == 1 ? reduced_coef(kind, n, side(r), c)
                                       : reduced_coef(kind, n, r, side(c));
        out[(((size_t)(r / 16) * kb[part] + c / 4) * 4 + c % 4) * 16 + r % 16] = v;
      }
  }
  return f;
}

void launch_mfma(hipStream_t s, int kind, int n, const R2RJob *jobs, int njob, double scale, const double *frag) {
  const MSplit m = mfma_split(kind, n);
  MArgs a{};
  a.scale = scale;
  a.n = n;
  a.half = m.half; a.rows = m.rows; a.ks = m.ks; a.ka = m.ka; a.na = m.na; a.hc = m.hc;
  a.ld = mfma_ld(m);
  a.ntile = (m.rows + 15) / 16;
  a.fs = frag;
  a.fa = frag + (size_t)a.ntile * ((m.ks + 3) / 4) * 64;
  // a wavefront per tile of rows up to eight; short lines get more line
  // groups per workgroup instead (at least four wavefronts)
  a.tw = std::min(a.ntile, 8);
  a.lg = a.tw == 1 ? 4 : (a.tw == 2 ? 2 : 1);
  long total = 0;
  for (int q = 0; q < njob; q++) total += (long)jobs[q].nb1 * jobs[q].nb2;
  // two tiles of lines per wavefront (each matrix load used twice) where two
  // workgroups still fit a CU's LDS and the launch has two workgroups per CU
  const int ntl = mfma_lds(a.ld, 32 * a.lg) <= LDS_MAX / 2 && total >= 32L * a.lg * 512 ? 2 : 1;
  while (a.lg > 1 && mfma_lds(a.ld, 16 * ntl * a.lg) > LDS_MAX) a.lg >>= 1;
  const int L = 16 * ntl * a.lg;
  int wg = 0;
  for (int q = 0; q < njob; q++) {
    const R2RJob &b = jobs[q];
    const int nlines = b.nb1 * b.nb2;
    if (nlines <= 0) continue;
    a.job[a.njob++] = MJob{b.in, b.out, b.ies, b.is1, b.is2, b.oes, b.os1, b.os2, b.nb1, nlines, wg};
    wg += (nlines + L - 1) / L;
  }
  if (wg == 0) return;
  const dim3 grid((unsigned)wg), blk(64 * a.tw * a.lg);
  const size_t lds = mfma_lds(a.ld, L);
  const bool sw = jobs[0].oes == 1;  // the same axis, so the same for every job
#define SNAC_MF(M, W, T) hipLaunchKernelGGL((k_r2r_mfma<M, W, T>), grid, blk, lds, s, a)
#define SNAC_MFM(M)                                                                  \
  do {                                                                               \
    if (sw) { if (ntl == 2) SNAC_MF(M, true, 2); else SNAC_MF(M, true, 1); }         \
    else { if (ntl == 2) SNAC_MF(M, false, 2); else SNAC_MF(M, false, 1); }          \
  } while (0)
  if (m.mode == 0) SNAC_MFM(0);
  else if (m.mode == 1) SNAC_MFM(1);
  else SNAC_MFM(2);
#undef SNAC_MFM
#undef SNAC_MF
}

std::mutex g_mu;
std::map<std::pair<int, int>, std::pair<R2RPlan, double *>> g_plans;

bool fft_kind(int kind) {
  return kind == K_R2HC || kind == K_HC2R || kind == K_REDFT10 || kind == K_REDFT01 || kind == K_RODFT10 ||
         kind == K_RODFT01;
}

}  // namespace

double r2r_coef(int kind, int n, int k, int j) {
  const double pi = std::acos(-1.0);
  switch (kind) {
  case K_R2HC:
    if (k <= n / 2) return std::cos(2.0 * pi * (double)j * k / n);
    return -std::sin(2.0 * pi * (double)j * (n - k) / n);
  case K_HC2R:
    if (j == 0) return 1.0;
    if (n % 2 == 0 && j == n / 2) return (k % 2) ? -1.0 : 1.0;
    if (j < (n + 1) / 2) return 2.0 * std::cos(2.0 * pi * (double)j * k / n);
    return -2.0 * std::sin(2.0 * pi * (double)(n - j) * k / n);
  case K_REDFT10: return 2.0 * std::cos(pi * (j + 0.5) * k / n);
  case K_REDFT01: return j == 0 ? 1.0 : 2.0 * std::cos(pi * j * (k + 0.5) / n);
  case K_RODFT10: return 2.0 * std::sin(pi * (j + 0.5) * (k + 1) / n);
  case K_RODFT01: return j == n - 1 ? ((k % 2) ? -1.0 : 1.0) : 2.0 * std::sin(pi * (j + 1) * (k + 0.5) / n);
  case K_REDFT11: return 2.0 * std::cos(pi * (j + 0.5) * (k + 0.5) / n);
  case K_RODFT11: return 2.0 * std::sin(pi * (j + 0.5) * (k + 0.5) / n);
  // DST-I: the transform of a staggered Dirichlet-Dirichlet axis (fft.f90:130-133)
  case K_RODFT00: return 2.0 * std::sin(pi * (j + 1) * (k + 1) / (n + 1));
  default: throw std::runtime_error("unsupported r2r kind " + std::to_string(kind));
  }
}

int r2r_tile_choices(const R2RPlan &pl) {
  if (!pl.fft) return 1;
  if (pl.mixed) return 2;
  return (pl.kind == K_R2HC || pl.kind == K_HC2R) && pl.n >= 8 ? 8 : 3;
}

R2RPlan r2r_plan(int kind, int n, bool rowwise) {
  std::lock_guard<std::mutex> lk(g_mu);
  auto key = std::make_pair(rowwise ? kind + 16 : kind, n);
  auto it = g_plans.find(key);
  if (it != g_plans.end()) return it->second.first;
  if (n < 1) throw std::runtime_error("r2r: invalid length");
  R2RPlan pl;
  pl.n = n;
  pl.kind = kind;
  pl.fft = fft_kind(kind) && n >= 4 && (n & (n - 1)) == 0 && n <= 1024;
  int m1, m2;
  if (!rowwise && (kind == K_R2HC || kind == K_HC2R) && rfft_mixed_split(n, m1, m2)) pl.fft = pl.mixed = true;
  std::vector<double> h;
  const double pi = std::acos(-1.0);
  if (pl.fft) {
    h.resize(4 * (size_t)n);
    for (int m = 0; m < n; m++) {
      h[2 * m] = std::cos(-2.0 * pi * m / n);
      h[2 * m + 1] = std::sin(-2.0 * pi * m / n);
    }
    for (int k = 0; k < n; k++) {
      h[2 * n + 2 * k] = std::cos(pi * k / (2.0 * n));
      h[2 * n + 2 * k + 1] = std::sin(pi * k / (2.0 * n));
    }
  } else {
    if (n > 2048) throw std::runtime_error("r2r: length " + std::to_string(n) + " needs the FFT path (power of two)");
    (void)r2r_coef(kind, n, 0, 0);  // refuses unknown kinds
    pl.mfma = !rowwise && mfma_fits(kind, n);
    if (pl.mfma) {
      h = mfma_fragments(kind, n);
    } else {
      h.resize((size_t)n * n);
      for (int k = 0; k < n; k++)
        for (int j = 0; j < n; j++) h[(size_t)k * n + j] = r2r_coef(kind, n, k, j);
    }
  }
  double *d = nullptr;
  SNAC_HIP(hipMalloc(&d, h.size() * sizeof(double)));
  SNAC_HIP(hipMemcpy(d, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice));
  pl.tab = d;
  g_plans[key] = {pl, d};
  return pl;
}

namespace {
// the jobs of one plan in one launch (matrix products: any, up to
// GRID_BLOCKS; else the same extents and strides, up to R2R_FIELDS)
void launch_jobs(hipStream_t s, const R2RPlan &pl, const R2RJob *jobs, int njob, double scale) {
  if (pl.mfma) {
    launch_mfma(s, pl.kind, pl.n, jobs, njob, scale, pl.tab);
    SNAC_HIP(hipGetLastError());
    return;
  }
  const R2RJob &j0 = jobs[0];
  Args a;
  a.in = j0.in; a.out = j0.out;
  for (int f = 0; f < njob; f++) {
    a.in = std::min(a.in, jobs[f].in);
    a.out = std::min(a.out, jobs[f].out);
  }
  for (int f = 0; f < R2R_FIELDS; f++) {
    a.fin[f] = f < njob ? jobs[f].in - a.in : 0;
    a.fout[f] = f < njob ? jobs[f].out - a.out : 0;
  }
  a.ies = j0.ies; a.is1 = j0.is1; a.is2 = j0.is2; a.oes = j0.oes; a.os1 = j0.os1; a.os2 = j0.os2;
  a.n = pl.n;
  a.logn = 0;
  while ((1 << a.logn) < pl.n) a.logn++;
  a.nb1 = j0.nb1;
  a.nf = j0.nb1 * j0.nb2;
  a.nlines = a.nf * njob;
  a.coal = (a.ies != 1) ? 1 : 0;
  if (a.nlines <= 0) return;
  if (pl.mixed) {
    int n1 = 0, n2 = 0;
    rfft_mixed_split(pl.n, n1, n2);
    const int ls = pl.lshift == 1 ? 1 : 0, L = std::max(1, rfft_lines(n1, n2) >> ls);
    a.L = L;
    a.scale = scale;
    a.tab = pl.tab;
    launch_rfft_mixed(pl.kind == K_HC2R, pl.n, ls, dim3((unsigned)((a.nlines + L - 1) / L)),
                      (size_t)L * (pl.n + RPAD) * sizeof(double), s, a);
  } else if (pl.fft && (pl.kind == K_R2HC || pl.kind == K_HC2R) && pl.n >= 8) {
    int n1 = 0, n2 = 0;
    fft_split(pl.n / 2, n1, n2);
    const int ls = pl.lshift <= 2 ? pl.lshift : 0, tpb = rfft_tpb(pl.lshift);
    const int L = std::max(1, rfft_lines(n1, n2) >> ls);  // the kernel's compile-time line count
    a.L = L;
    a.scale = scale;
    a.tab = pl.tab;
    const int ntile = (a.nlines + L - 1) / L;
    dim3 grid((unsigned)((ntile + tpb - 1) / tpb));
    size_t lds = (size_t)L * (pl.n + RPAD) * sizeof(double);
    launch_rfft(pl.kind == K_HC2R, pl.n, pl.lshift, grid, lds, s, a);
  } else if (pl.fft) {
    int n1 = 0, n2 = 0;
    fft_split(pl.n, n1, n2);
    const int ls = pl.lshift <= 2 ? pl.lshift : 0;
    const int L = std::max(1, fft_lines(n1, n2) >> ls);  // the kernel's compile-time line count
    a.L = L;
    a.scale = scale;
    a.tab = pl.tab;
    dim3 grid((unsigned)((a.nlines + L - 1) / L));
    size_t lds = (size_t)L * pl.n * sizeof(double2);
    launch_fft_kind(pl.kind, pl.n, ls, grid, lds, s, a);
  } else {
    int L = std::max(1, std::min(2 * LDS_COMPLEX / pl.n, a.nlines));
    a.L = L;
    a.scale = scale;
    a.tab = pl.tab;
    dim3 grid((a.nlines + L - 1) / L);
    size_t lds = (size_t)L * pl.n * sizeof(double);
    hipLaunchKernelGGL(k_r2r_dense, grid, dim3(NT), lds, s, a);
  }
  SNAC_HIP(hipGetLastError());
}

}  // namespace

void launch_r2r(hipStream_t s, const R2RPlan &pl, const double *in, long ies, long is1, long is2, double *out,
                long oes, long os1, long os2, int nb1, int nb2, double scale) {
  const R2RJob j{in, ies, is1, is2, out, oes, os1, os2, nb1, nb2};
  launch_jobs(s, pl, &j, 1, scale);
}

void launch_r2r_jobs(hipStream_t s, const R2RPlan &pl, const std::vector<R2RJob> &jobs, double scale) {
  auto alike = [](const R2RJob &x, const R2RJob &y) {
    return x.ies == y.ies && x.is1 == y.is1 && x.is2 == y.is2 && x.oes == y.oes && x.os1 == y.os1 && x.os2 == y.os2 &&
           x.nb1 == y.nb1 && x.nb2 == y.nb2;
  };
  // the dense kernel keeps its launch per batch of lines
  const size_t most = pl.mfma ? GRID_BLOCKS : (pl.fft ? R2R_FIELDS : 1);
  for (size_t q = 0; q < jobs.size();) {
    size_t e = q + 1;
    while (e < jobs.size() && e - q < most && (pl.mfma || alike(jobs[q], jobs[e]))) e++;
    launch_jobs(s, pl, &jobs[q], (int)(e - q), scale);
    q = e;
  }
}

}  // namespace snac
