// Partitioned column solver on the level-fastest layout: scalar rows and 2x2
// and 3x3 block rows, everything of a column kept on chip.
//
// S lanes of a wavefront share a column, lane s holding its rows s*M ..
// s*M+M-1.  Each lane eliminates its rows but the last in registers,
//   x(e) = y(e) - g(e) x(e+1) - h(e) xl      (xl: the previous lane's last row),
// which leaves one row per lane; the S of them are solved by cyclic reduction
// across the lanes, and the lane's other rows follow by substitution.
//
// What bounds it: HBM for scalar rows; for block rows chains of dependent FP64
// instructions in the one or two wavefronts per SIMD that their registers leave
// room for (the VALU busy 42% of the time on 2x2 rows, 27% on 3x3).
// Every coefficient is read once and every unknown written once.  A thread per
// column, or a wavefront per column reduced row by row (the solvers before),
// kept ratios or block gammas in HBM between two sweeps, read each array with
// a stride of a whole column, or spent seven exchanges of whole rows.  Here a
// wavefront loads its 64/S columns in runs of 64 consecutive doubles, all
// loads in flight at once, and turns each array round through LDS to the lanes
// that own the rows (one padding double per lane makes the stride odd: no bank
// conflicts).  Measured, before and after (a plain copy moves 4.9 TB/s):
//   scalar, 165,888 columns x 112 rows   359 ->  148 us (5.0 TB/s)
//   2x2,     41,472 columns x 112 rows   755 ->  146 us (4.1 TB/s)
//   3x3,     10,368 columns x  56 rows   475 ->   76 us (2.0 TB/s)
// Staging whole columns in LDS instead of registers: 206, 418 and 149 us (two
// to five wavefronts per CU).
//
// Rows per lane M, lanes per column S: more rows per lane mean fewer reduction
// steps and less rounding (scalar, relative error 2.4e-16 with M = 8, 2.6e-16
// with 4, 2.9e-16 reduced row by row), and more registers for y, g and h.
// Scalar rows take M = 4 and 8 or 16 lanes up to 64 rows (28 rows, 2,592, 10,368
// and 165,888 columns: 5.3, 6.4 and 32 us against 7.6, 8.4 and 40 with M = 8; 56
// rows, 2,592 and 41,472: 4.5 and 17 us against 6.1 and 19), beyond that M = 8,
// where DPP no longer reaches across a column of M = 4.  2x2 rows at M = 4 just fit two
// wavefronts per SIMD (113 levels, before the limits on multipliers were one
// comparison each: 168 us, 190 with M = 2); up to 32 rows
// M = 2 fits three (43 us against 48, 41,472 x 28).  3x3 rows at M = 4 use
// every register of a SIMD (56 rows: 78 us, 118 with M = 2), up to 32 rows
// M = 2 is as fast (41 and 48 us) and faster on few columns (14 and 23).
// Up to S = 16 the lanes exchange by DPP row shifts, no LDS traffic.
#include "tgx_common.h"

namespace tgx {
namespace seg {

// A lane's dword from the lane `d` below (up: above) in its 16-lane row, zero
// past the row's end.
template <int CTRL>
__device__ __forceinline__ double dpp_row(double v) {
  union { double d; int w[2]; } a, b;
  a.d = v;
  b.w[0] = __builtin_amdgcn_update_dpp(0, a.w[0], CTRL, 0xf, 0xf, true);
  b.w[1] = __builtin_amdgcn_update_dpp(0, a.w[1], CTRL, 0xf, 0xf, true);
  return b.d;
}
// The value of segment lane - D / lane + D of the column, 0 outside 0..S-1.
template <int S, int D>
__device__ __forceinline__ double from_below(double v, int lane) {
  if (S == 16) return dpp_row<0x110 + (D & 15)>(v);
  const double t = S < 16 ? dpp_row<0x110 + (D & 15)>(v) : __shfl(v, lane - D, S);
  return lane >= D ? t : 0.;
}
template <int S, int D>
__device__ __forceinline__ double from_above(double v, int lane) {
  if (S == 16) return dpp_row<0x100 + (D & 15)>(v);
  const double t = S < 16 ? dpp_row<0x100 + (D & 15)>(v) : __shfl(v, lane + D, S);
  return lane + D < S ? t : 0.;
}

// N x N blocks, column-major (element (r, c) at r + N*c), as the callers'.
template <int N>
struct Mat { double v[N * N]; };
template <int N>
struct Vec { double v[N]; };

template <int N>
__device__ __forceinline__ Mat<N> mul(const Mat<N> &a, const Mat<N> &b) {
  Mat<N> r;
#pragma unroll
  for (int c = 0; c < N; ++c)
#pragma unroll
    for (int i = 0; i < N; ++i) {
      double t = a.v[i] * b.v[N * c];
#pragma unroll
      for (int l = 1; l < N; ++l) t = __builtin_fma(a.v[i + N * l], b.v[l + N * c], t);
      r.v[i + N * c] = t;
    }
  return r;
}
// x - a b
template <int N>
__device__ __forceinline__ Mat<N> sub(const Mat<N> &x, const Mat<N> &a, const Mat<N> &b) {
  Mat<N> r = x;
#pragma unroll
  for (int c = 0; c < N; ++c)
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int l = 0; l < N; ++l) r.v[i + N * c] = __builtin_fma(-a.v[i + N * l], b.v[l + N * c], r.v[i + N * c]);
  return r;
}
template <int N>
__device__ __forceinline__ Vec<N> mul(const Mat<N> &a, const Vec<N> &b) {
  Vec<N> r;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    double t = a.v[i] * b.v[0];
#pragma unroll
    for (int l = 1; l < N; ++l) t = __builtin_fma(a.v[i + N * l], b.v[l], t);
    r.v[i] = t;
  }
  return r;
}
template <int N>
__device__ __forceinline__ Vec<N> sub(const Vec<N> &x, const Mat<N> &a, const Vec<N> &b) {
  Vec<N> r = x;
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int l = 0; l < N; ++l) r.v[i] = __builtin_fma(-a.v[i + N * l], b.v[l], r.v[i]);
  return r;
}
template <int N>
__device__ __forceinline__ Mat<N> neg(Mat<N> a) {
#pragma unroll
  for (int n = 0; n < N * N; ++n) a.v[n] = -a.v[n];
  return a;
}
template <int N>
__device__ __forceinline__ Mat<N> inverse(const Mat<N> &m) {
  Mat<N> r;
  const double *a = m.v;
  if (N == 1) {
    r.v[0] = 1. / a[0];
  } else if (N == 2) {
    const double d = 1. / __builtin_fma(a[0], a[3], -(a[2] * a[1]));
    r.v[0] = a[3] * d;
    r.v[1 % (N * N)] = -a[1] * d;
    r.v[2 % (N * N)] = -a[2] * d;
    r.v[3 % (N * N)] = a[0] * d;
  } else {
    auto M = [&](int i, int j) { return a[(i % 3) + 3 * (j % 3)]; };
    double co[9];
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int i = 0; i < 3; ++i)
        co[i + 3 * j] = __builtin_fma(M(i + 1, j + 1), M(i + 2, j + 2), -(M(i + 1, j + 2) * M(i + 2, j + 1)));
    const double d = 1. / __builtin_fma(a[0], co[0], __builtin_fma(a[3], co[3], a[6] * co[6]));
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int i = 0; i < 3; ++i) r.v[(j + 3 * i) % (N * N)] = co[i + 3 * j] * d;
  }
  return r;
}
// Whether an element of a is beyond lim, or not a number.
template <int N>
__device__ __forceinline__ bool beyond(const Mat<N> &a, double lim) {
  bool r = false;
#pragma unroll
  for (int n = 0; n < N * N; ++n) r |= !(fabs(a.v[n]) <= lim);
  return r;
}
template <int S, int D, class T>
__device__ __forceinline__ T below(const T &a, int lane) {
  T r;
#pragma unroll
  for (int n = 0; n < (int)(sizeof(T) / 8); ++n) r.v[n] = from_below<S, D>(a.v[n], lane);
  return r;
}
template <int S, int D, class T>
__device__ __forceinline__ T above(const T &a, int lane) {
  T r;
#pragma unroll
  for (int n = 0; n < (int)(sizeof(T) / 8); ++n) r.v[n] = from_above<S, D>(a.v[n], lane);
  return r;
}

// Multipliers beyond this mark a column whose segments are badly pivoted on
// their own (a diagonal block small beside its couplings, which Thomas never
// pivots on unreduced): it is refined (refine_columns).  Held
// against it are a row's multipliers and their products over the lane's rows, by
// which an error of one row reaches another: multipliers of 2 to 31 in a
// segment of eight scalar rows, all below a limit of 32 for each, lost 2 to 11
// digits.  Rows with diagonal dominance keep all of them at 1 or below.
// Emulated on columns without dominance, those within 4 have a median error 0.9
// to 1.4 times that of the reference's order (advection at Peclet numbers up to 3,
// random blocks plus once or twice the identity, 28 to 200 rows); within 32, with
// the products, up to 4.6 times.
constexpr double GROWTH = 4.;

// Cyclic reduction of x(s) + a x(s-1) + c x(s+1) = d over the S lanes of a
// column, unit diagonal blocks; the last step needs d only.  bad: a multiplier
// is beyond GROWTH.
template <int N, int S, int D>
__device__ __forceinline__ void reduce(Mat<N> &a, Mat<N> &c, Vec<N> &d, int lane, bool &bad) {
  const Mat<N> am = below<S, D>(a, lane), cm = below<S, D>(c, lane), ap = above<S, D>(a, lane),
               cp = above<S, D>(c, lane);
  const Vec<N> dm = below<S, D>(d, lane), dp = above<S, D>(d, lane);
  Mat<N> w = {};
#pragma unroll
  for (int n = 0; n < N; ++n) w.v[n * (N + 1)] = 1.;
  w = inverse(sub(sub(w, a, cm), c, ap));
  d = mul(w, sub(sub(d, a, dm), c, dp));
  if constexpr (2 * D < S) {
    a = neg(mul(w, mul(a, am)));
    c = neg(mul(w, mul(c, cp)));
    bad |= beyond(a, GROWTH) | beyond(c, GROWTH);
    reduce<N, S, 2 * D>(a, c, d, lane, bad);
  }
}

// Elimination in the reference's order over one column, by one lane: the
// ratios / gammas go to G, the solution to X (both LDS, n rows).  Scalar
// (trsolv.F:63-101), 2x2 (duv.F:830-906), 3x3 (comp_ng.F90:281-326).
template <int N>
__device__ __noinline__ void serial_column(const double *A, const double *B, const double *C, const double *F, double *G,
                                           double *X, int n) {
  double gam[9] = {}, y[3] = {};
  for (int k = 0; k < n; ++k) {
    double p[9], q[9], r[9], f[3], w[9];
    for (int e = 0; e < N * N; ++e) {
      p[e] = k ? A[k * N * N + e] : 0.;
      q[e] = B[k * N * N + e];
      r[e] = k < n - 1 ? C[k * N * N + e] : 0.;
    }
    for (int i = 0; i < N; ++i) f[i] = F[k * N + i];
    for (int m = 0; m < N; ++m)
      for (int l = 0; l < N; ++l)
        for (int i = 0; i < N; ++i) q[i + N * m] = q[i + N * m] - p[i + N * l] * gam[l + N * m];
    for (int m = 0; m < N; ++m)
      for (int i = 0; i < N; ++i) f[i] = f[i] - p[i + N * m] * y[m];
    if (N == 1) {
      gam[0] = r[0] / q[0];
      y[0] = f[0] / q[0];
    } else {
      if (N == 2) {
        const double d = q[0] * q[3] - q[2] * q[1];
        w[0] = q[3] / d;
        w[1] = -q[1] / d;
        w[2] = -q[2] / d;
        w[3] = q[0] / d;
      } else {
        const double d = q[0] * q[4] * q[8] - q[0] * q[7] * q[5] - q[3] * q[1] * q[8] + q[3] * q[7] * q[2] +
                         q[6] * q[1] * q[5] - q[6] * q[4] * q[2];
        w[0] = (q[4] * q[8] - q[7] * q[5]) / d;
        w[1] = -(q[1] * q[8] - q[7] * q[2]) / d;
        w[2] = (q[1] * q[5] - q[4] * q[2]) / d;
        w[3] = -(q[3] * q[8] - q[6] * q[5]) / d;
        w[4] = (q[0] * q[8] - q[6] * q[2]) / d;
        w[5] = -(q[0] * q[5] - q[3] * q[2]) / d;
        w[6] = (q[3] * q[7] - q[6] * q[4]) / d;
        w[7] = -(q[0] * q[7] - q[6] * q[1]) / d;
        w[8] = (q[0] * q[4] - q[3] * q[1]) / d;
      }
      for (int m = 0; m < N; ++m)
        for (int i = 0; i < N; ++i) {
          double t = 0.;
          for (int l = 0; l < N; ++l) t = t + w[i + N * l] * r[l + N * m];
          gam[i + N * m] = t;
        }
      for (int i = 0; i < N; ++i) {
        double t = 0.;
        for (int m = 0; m < N; ++m) t = t + w[i + N * m] * f[m];
        y[i] = t;
      }
    }
    for (int e = 0; e < N * N; ++e) G[k * N * N + e] = gam[e];
    for (int i = 0; i < N; ++i) X[k * N + i] = y[i];
  }
  for (int k = n - 2; k >= 0; --k) {
    double x[3];
    for (int i = 0; i < N; ++i) {
      x[i] = X[k * N + i];
      for (int m = 0; m < N; ++m) x[i] = x[i] - G[k * N * N + i + N * m] * y[m];
    }
    for (int i = 0; i < N; ++i) X[k * N + i] = y[i] = x[i];
  }
}

// The largest correction of a block row, relative to the largest unknown of the
// row and its neighbours, that is rounding: 1e-15 on dominant rows, 7e-14 where
// the dominance is 1e-5 to 1e-3 (56 to 200 rows), 1e-12 for a solution that falls
// by a decade per row; 1e-11 where a segment lost five digits.
constexpr double CORRECTION = 1e-12;
// A badly pivoted column is refined: the same elimination solves for the
// residual, which is computed in 64 bits from the rows themselves.  A first
// correction within REFINED of the unknowns shows that the elimination keeps
// eight digits, so that what it leaves is below rounding.  A later one shows
// less (each correction is an elimination's error further down, and where
// products of multipliers pass 1e10 that error stops falling as rounding itself is
// multiplied), so it has to be within SETTLED.  With 1e-8 for those too, pivots of
// 1e-2 in segments of eight rows kept errors of 3e-12; now 6e-14 at most (reduced
// row by row 8e-14, the reference's order 2e-14).  At most REFINEMENTS
// times, then in the reference's order by one lane, as where a pivot
// vanished and nothing finite came out.  Emulated on the families above, one
// pass suffices but for multipliers of 20 and more over eight rows (two) and 1
// in 100 random 3x3 columns (three); the error is 0.2 to 0.9 times that of the
// reference's order.  One lane per column for all of them instead: scalar
// 165,888 x 112, every column bad, 1,280 us; 2x2 41,472 x 112 1,660; 3x3 10,368 x
// 56 520; refined 361, 257 to 285 and 136 (a wavefront per column reduced row by row, or a
// thread per column, took 355, 577 and 337).
constexpr double REFINED = 1e-8, SETTLED = 1e-13;
constexpr int REFINEMENTS = 3;

// The rows of a block's nc columns, column c0 the first: 64 consecutive doubles
// per load, every load in flight at once, then through LDS (sm) to the lanes
// that own the rows, one array after the other.  Identity rows past the column.
template <int N, int S, int M>
__device__ __forceinline__ void load_rows(int t, const double *a, const double *b, const double *c, const double *f,
                                          long c0, int nc, int ldk, int n, double *sm, Mat<N> (&A)[M], Mat<N> (&B)[M],
                                          Mat<N> (&Cm)[M], Vec<N> (&F)[M]) {
  constexpr int C = 64 / S, NN = N * N;
  constexpr int QM = (S * M * NN + 63) / 64, QV = (S * M * N + 63) / 64;  // loads of one column
  double va[C * QM], vb[C * QM], vc[C * QM], vf[C * QV];
#define SEG_LOAD(buf, src, per, Q)                                                                          \
  _Pragma("unroll") for (int cc = 0; cc < C; ++cc) _Pragma("unroll") for (int q = 0; q < Q; ++q)          \
      if (cc < nc && 64 * q + t < n * (per)) buf[cc * Q + q] = src[(size_t)(c0 + cc) * ldk * (per) + (64 * q + t)];
  SEG_LOAD(va, a, NN, QM)
  SEG_LOAD(vb, b, NN, QM)
  SEG_LOAD(vc, c, NN, QM)
  SEG_LOAD(vf, f, N, QV)
#undef SEG_LOAD
  const bool col = t / S < nc;
  const int r0 = t % S * M;
#define SEG_ROWS(dst, buf, per, Q, on, other)                                                               \
  _Pragma("unroll") for (int cc = 0; cc < C; ++cc) _Pragma("unroll") for (int q = 0; q < Q; ++q)          \
      if (64 * q + t < S * M * (per)) sm[cc * S * (M * (per) + 1) + (64 * q + t) + (64 * q + t) / (M * (per))] = buf[cc * Q + q]; \
  __syncthreads();                                                                                        \
  _Pragma("unroll") for (int e = 0; e < M; ++e) _Pragma("unroll") for (int q = 0; q < (per); ++q) {       \
    const double w = sm[t * (M * (per) + 1) + e * (per) + q];                                             \
    dst[e].v[q] = col && (on) ? w : (other);                                                              \
  }                                                                                                       \
  __syncthreads();
  SEG_ROWS(A, va, NN, QM, r0 + e > 0 && r0 + e < n, 0.)
  SEG_ROWS(B, vb, NN, QM, r0 + e < n, q % (N + 1) == 0 ? 1. : 0.)
  SEG_ROWS(Cm, vc, NN, QM, r0 + e < n - 1, 0.)
  SEG_ROWS(F, vf, N, QV, r0 + e < n, 0.)
#undef SEG_ROWS
}

// The partitioned elimination: xs the lane's unknowns, xl the previous lane's
// last one; bad: a multiplier or a product of them is beyond GROWTH.
template <int N, int S, int M>
__device__ __forceinline__ void eliminate(const Mat<N> (&A)[M], const Mat<N> (&B)[M], const Mat<N> (&Cm)[M],
                                          const Vec<N> (&F)[M], int lane, Vec<N> (&xs)[M], Vec<N> &xl, bool &bad) {
  Mat<N> g[M - 1], h[M - 1];
  Vec<N> y[M - 1];
  bad = false;
#pragma unroll
  for (int e = 0; e < M - 1; ++e) {
    if (e == 0) {
      const Mat<N> I = inverse(B[0]);
      g[0] = mul(I, Cm[0]);
      h[0] = mul(I, A[0]);
      y[0] = mul(I, F[0]);
    } else {
      const Mat<N> I = inverse(sub(B[e], A[e], g[e - 1]));
      g[e] = mul(I, Cm[e]);
      h[e] = neg(mul(I, mul(A[e], h[e - 1])));
      y[e] = mul(I, sub(F[e], A[e], y[e - 1]));
    }
    bad |= beyond(g[e], GROWTH) | beyond(h[e], GROWTH);
  }
  // the lane's first row in its last row and xl, for the lane before
  Vec<N> Y = y[M - 2], X;
  Mat<N> G = g[M - 2], H = h[M - 2];
#pragma unroll
  for (int e = M - 3; e >= 0; --e) {
    Y = sub(y[e], g[e], Y);
    H = sub(h[e], g[e], H);
    G = neg(mul(g[e], G));
    bad |= beyond(G, GROWTH) | beyond(H, GROWTH);
  }
  {
    const Vec<N> Yn = above<S, 1>(Y, lane);
    const Mat<N> Gn = above<S, 1>(G, lane), Hn = above<S, 1>(H, lane);
    const Mat<N> I = inverse(sub(sub(B[M - 1], A[M - 1], g[M - 2]), Cm[M - 1], Hn));
    Mat<N> ra = neg(mul(I, mul(A[M - 1], h[M - 2]))), rc = neg(mul(I, mul(Cm[M - 1], Gn)));
    X = mul(I, sub(sub(F[M - 1], A[M - 1], y[M - 2]), Cm[M - 1], Yn));
    bad |= beyond(ra, GROWTH) | beyond(rc, GROWTH);
    reduce<N, S, 1>(ra, rc, X, lane, bad);
  }
  xl = below<S, 1>(X, lane);
  xs[M - 1] = X;
#pragma unroll
  for (int e = M - 2; e >= 0; --e) xs[e] = sub(sub(y[e], h[e], xl), g[e], xs[e + 1]);
}

// The largest unknown of a row and its neighbours.
template <int N>
__device__ __forceinline__ double largest(const Vec<N> &p, const Vec<N> &q, const Vec<N> &r) {
  double big = 0.;
#pragma unroll
  for (int n = 0; n < N; ++n) big = fmax(fmax(big, fabs(p.v[n])), fmax(fabs(q.v[n]), fabs(r.v[n])));
  return big;
}

// Stores the columns whose lanes are in `done` from the lanes' rows in sv.
template <int N, int S, int M>
__device__ __forceinline__ void store_columns(unsigned long long done, double *x, long c0, int ldk, int n,
                                              const double *sv) {
  constexpr int C = 64 / S, LV = M * N + 1, QV = (S * M * N + 63) / 64;
#pragma unroll
  for (int cc = 0; cc < C; ++cc)
    if (done >> (cc * S) & 1)
#pragma unroll
      for (int q = 0; q < QV; ++q) {
        const int e = 64 * q + (int)threadIdx.x;
        if (e < n * N) x[(size_t)(c0 + cc) * ldk * N + e] = sv[cc * S * LV + e + e / (M * N)];
      }
}

// The columns whose lanes are in todo, badly pivoted, their first solution in sv.
template <int N, int S, int M>
__device__ __forceinline__ void refine_columns(const double *a, const double *b, const double *c, const double *f,
                                            double *x, int ldk, int n, long c0, int nc, double *sm, double *sv,
                                            unsigned long long todo) {
  constexpr int NN = N * N, LM = M * NN + 1, LV = M * N + 1;
  unsigned long long serial = 0;
  int t = threadIdx.x;
  // the solution so far, rows -1 and M from the neighbouring lanes
  auto solved = [&](int e) {
    const int lane = t % S;
    Vec<N> r;
    const bool in = (e >= 0 || lane > 0) && (e < M || lane + 1 < S);
    const int o = !in ? 0 : e < 0 ? (t - 1) * LV + (M - 1) * N : e < M ? t * LV + e * N : (t + 1) * LV;
#pragma unroll
    for (int q = 0; q < N; ++q) r.v[q] = in ? sv[o + q] : 0.;
    return r;
  };
#pragma unroll 1
  for (int pass = 0; pass < REFINEMENTS && todo; ++pass) {
    asm volatile("" : "+v"(t));  // addresses formed anew in every pass: the registers are the rows'
    const int lane = t % S;
    const unsigned long long own = (S == 64 ? ~0ull : (1ull << (S & 63)) - 1) << (t / S * S & 63);  // this column's lanes
    Mat<N> A[M], B[M], Cm[M];
    Vec<N> F[M], d[M], dl;
    load_rows<N, S, M>(t, a, b, c, f, c0, nc, ldk, n, sm, A, B, Cm, F);
#pragma unroll
    for (int e = 0; e < M; ++e) {
      F[e] = sub(sub(sub(F[e], A[e], solved(e - 1)), B[e], solved(e)), Cm[e], solved(e + 1));
      asm volatile("" ::: "memory");  // read again below: the registers are the elimination's
    }
    bool bad;
    eliminate<N, S, M>(A, B, Cm, F, lane, d, dl, bad);
    bad = false;
    bool lost = false;  // nothing to refine
#pragma unroll
    for (int e = 0; e < M; ++e) {
      asm volatile("" ::: "memory");
      const Vec<N> here = solved(e);
      const double big = largest(solved(e - 1), here, solved(e + 1));
#pragma unroll
      for (int q = 0; q < N; ++q) {
        bad |= !(fabs(d[e].v[q]) <= (pass ? SETTLED : REFINED) * big);
        d[e].v[q] = here.v[q] + d[e].v[q];
        lost |= !(fabs(d[e].v[q]) <= 1.e300);
      }
    }
    __syncthreads();  // the neighbours have read this lane's solution
#pragma unroll
    for (int e = 0; e < M; ++e)
#pragma unroll
      for (int q = 0; q < N; ++q) sv[t * LV + e * N + q] = d[e].v[q];
    __syncthreads();
    const unsigned long long bads = __ballot(bad), losts = __ballot(lost);
    serial |= __ballot((losts & own) != 0) & todo;
    const unsigned long long again = __ballot((bads & own) != 0) & todo & ~serial;
    store_columns<N, S, M>(todo & ~serial & ~again, x, c0, ldk, n, sv);
    todo = again;
  }
  serial |= todo;
  if (!serial) return;
  __syncthreads();
  const int cw = t / S;
  if (t % S == 0 && (serial >> t & 1)) {
    const size_t o = (size_t)(c0 + cw) * ldk;
    serial_column<N>(a + o * NN, b + o * NN, c + o * NN, f + o * N, sm + cw * S * LM, sv + cw * S * LV, n);
    for (int e = 0; e < n * N; ++e) x[o * N + e] = sv[cw * S * LV + e];
  }
}

template <int N, int S, int M>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(N == 1 ? (M == 4 ? 6 : S == 16 ? 5 : 4) : N == 3 ? 1 : M == 2 ? 3 : 2)))
segment_kernel(const double *__restrict__ a, const double *__restrict__ b, const double *__restrict__ c,
               const double *f, double *x, int ldk, int n, int ncol) {
  constexpr int C = 64 / S, LV = M * N + 1;
  __shared__ double sm[64 * (M * N * N + 1)], sv[64 * LV];  // a lane's rows and one double of padding
  const int t = threadIdx.x, lane = t % S, cw = t / S;
  const long c0 = (long)tgx_xcd_block(gridDim.x) * C;
  const int nc = (int)min((long)C, ncol - c0);  // at least 1
  Mat<N> A[M], B[M], Cm[M];
  Vec<N> F[M], xs[M], xl;
  load_rows<N, S, M>(t, a, b, c, f, c0, nc, ldk, n, sm, A, B, Cm, F);
  bool bad;
  eliminate<N, S, M>(A, B, Cm, F, lane, xs, xl, bad);
  if (N > 1) {
    // One correction of each row from its neighbours, x(k) += B^-1 (F - A
    // x(k-1) - B x(k) - C x(k+1)): takes the rounding of the two extra
    // substitutions of a partitioned solve back out (relative error 1.0e-16
    // on dominant 2x2 rows and 1.1e-16 on 3x3, 2.0e-16 and 2.4e-16 without;
    // Thomas 1.5e-16 and 1.8e-16).  It is also the proof of the solution: a
    // column with a correction beyond CORRECTION is solved again.
    const Vec<N> xn = above<S, 1>(xs[0], lane);
    Vec<N> prev = xl;
#pragma unroll
    for (int e = 0; e < M; ++e) {
      const Vec<N> next = e < M - 1 ? xs[e < M - 1 ? e + 1 : 0] : xn, here = xs[e];
      const Vec<N> r = mul(inverse(B[e]), sub(sub(sub(F[e], A[e], prev), B[e], here), Cm[e], next));
      const double big = largest(prev, here, next);
#pragma unroll
      for (int q = 0; q < N; ++q) {
        bad |= !(fabs(r.v[q]) <= CORRECTION * big);
        xs[e].v[q] = here.v[q] + r.v[q];
      }
      prev = here;
    }
  }
#pragma unroll
  for (int e = 0; e < M; ++e)
#pragma unroll
    for (int q = 0; q < N; ++q) sv[t * LV + e * N + q] = xs[e].v[q];
  __syncthreads();
  const unsigned long long own = (S == 64 ? ~0ull : (1ull << (S & 63)) - 1) << (cw * S & 63);
  const unsigned long long all = __ballot(cw < nc), vote = __ballot(bad), todo = __ballot((vote & own) != 0) & all;
  store_columns<N, S, M>(all & ~todo, x, c0, ldk, n, sv);
  if (todo) refine_columns<N, S, M>(a, b, c, f, x, ldk, n, c0, nc, sm, sv, todo);
}

template <int N, int S, int M>
int launch(const double *a, const double *b, const double *c, const double *f, double *x, int ldk, int n, int ncol,
           hipStream_t s) {
  constexpr int C = 64 / S;
  const int nb = (int)(((long)ncol + C - 1) / C);
  hipLaunchKernelGGL((segment_kernel<N, S, M>), dim3(nb), dim3(64), 0, s, a, b, c, f, x, ldk, n, ncol);
  TGX_HIP(hipGetLastError());
  return 0;
}

}  // namespace seg
}  // namespace tgx

// n rows (at most 256) of ncol columns, column j's rows from element 0 of
// a + j*ldk*nblk^2 (b, c alike), f + j*ldk*nblk, x + j*ldk*nblk.
extern "C" int tgx_launch_segment(int nblk, const double *a, const double *b, const double *c, const double *f,
                                  double *x, int ldk, int n, int ncol, hipStream_t s) {
  using namespace tgx::seg;
  if (ncol <= 0 || n <= 0) return 0;
  if (n > 256) return tgx_set_error(1, "the partitioned solver holds at most 256 rows per column (got %d)", n);
  if (nblk == 1) {
    if (n <= 32) return launch<1, 8, 4>(a, b, c, f, x, ldk, n, ncol, s);
    if (n <= 64) return launch<1, 16, 4>(a, b, c, f, x, ldk, n, ncol, s);
    if (n <= 128) return launch<1, 16, 8>(a, b, c, f, x, ldk, n, ncol, s);
    return launch<1, 32, 8>(a, b, c, f, x, ldk, n, ncol, s);
  }
  if (nblk == 2) {
    if (n <= 32) return launch<2, 16, 2>(a, b, c, f, x, ldk, n, ncol, s);
    if (n <= 64) return launch<2, 16, 4>(a, b, c, f, x, ldk, n, ncol, s);
    if (n <= 128) return launch<2, 32, 4>(a, b, c, f, x, ldk, n, ncol, s);
    return launch<2, 64, 4>(a, b, c, f, x, ldk, n, ncol, s);
  }
  if (n <= 32) return launch<3, 16, 2>(a, b, c, f, x, ldk, n, ncol, s);
  if (n <= 64) return launch<3, 16, 4>(a, b, c, f, x, ldk, n, ncol, s);
  if (n <= 128) return launch<3, 32, 4>(a, b, c, f, x, ldk, n, ncol, s);
  return launch<3, 64, 4>(a, b, c, f, x, ldk, n, ncol, s);
}
