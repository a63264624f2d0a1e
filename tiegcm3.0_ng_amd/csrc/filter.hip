// The high-latitude longitude ring filter of the global model
// (ringfilter.F:1-111), applied after the column solves of dt, duv, minor,
// comp and oplus (filter_tn dt.F:431-511 and its siblings) to the latitudes
// next to each pole.  A wavefront filters one level of one latitude row at a
// time: the row's longitudes in registers, the Fourier coefficients of the
// kept harmonics as wavefront reductions over a table of cos(m ang) and
// sin(m ang) (the only transcendental work), the residual and the chunk
// averages in its own LDS region.  Two forms of the launch:
//  - tgx_ringfilter_dev and the host drop-in: a block of eight wavefronts
//    takes eight levels of one row and first builds the table in LDS;
//  - the global routines (tgx_ringfilter_post_dev): the table is built once
//    per call in the workspace, a block is one wavefront and one level (small
//    blocks that find room beside the other routines' column kernels), all
//    the routine's fields go in one launch, and the routine's post pass (time
//    smoothing, top level, floors) is applied to each filtered value as it is
//    written.
#include <hip/hip_runtime.h>

#include "../../include/tgx.h"
#include "tgx_common.h"

namespace tgx {
namespace ring {

constexpr int kMaxOrder = TGX_RING_MAX_ORDER;
constexpr int kLdsMax = 65536;  // dynamic LDS of one block
// Wavefronts of a block of the LDS-table form: they share one table (at 576
// longitudes and order 3, 27 KB and 3.4 sincos per thread), and two blocks of
// eight fit in a CU.  0.625 deg, 80 rows of 113 levels: 44 us with eight, 53
// with four, 64 with two.
constexpr int kWaves = 8;
static_assert(64 * 32 >= TGX_RING_MAX_NLON, "ringfilter_kernel<32> covers the longest row");

// The rows of one launch, by value in the kernel arguments: row r is at
// f + k * plane + off[r] and is filtered with n[r] chunks.
struct Rows {
  long off[TGX_RING_MAX_ROWS];
  int n[TGX_RING_MAX_ROWS];
};

// The post pass that follows the filter in each global routine, on the
// filtered latitudes: dt.F:396-424 (POST_DT), duv.F:501-514 (POST_DUV),
// minor.F:556-597 (POST_MINOR), oplus.F:911-934 (POST_OPLUS).
enum PostKind { POST_NONE = 0, POST_DT, POST_DUV, POST_MINOR, POST_OPLUS };
constexpr double DTSMOOTH = 0.95, DTSMOOTH_DIV2 = 0.5 * (1. - DTSMOOTH), SPVAL = 1.e36;

// The fields of one launch: f[q] is filtered in place on levels 0..nlev-1;
// with a post pass, xnm[q] receives the n-1 field from the step inputs fin[q]
// (n) and fnmi[q] (n-1), and a level nlev < nk (the top) is set to spval or
// zero without filtering.
struct Fields {
  double *f[4], *xnm[4];
  const double *fin[4], *fnmi[4];
  int nf, nlev, kind;
};

// The post pass of one filtered value y with the step inputs fi (n) and fm
// (n-1): the solution xo and the n-1 field xn, in the reference's order.
__device__ __forceinline__ void post_point(int kind, double y, double fi, double fm, double &xo, double &xn) {
  if (kind == POST_DT) {
    xn = DTSMOOTH_DIV2 * (fm + y) + DTSMOOTH * fi;
    xo = y < 100. ? 100. : y;
  } else if (kind == POST_DUV) {
    xn = DTSMOOTH_DIV2 * (fm + y) + DTSMOOTH * fi;
    xo = y;
  } else if (kind == POST_MINOR) {
    const double small = 1.e-12;
    const double nm = DTSMOOTH * fi + DTSMOOTH_DIV2 * (fm + y);
    xo = y < small ? small : y;
    xn = nm < small ? small : nm;
  } else {  // POST_OPLUS
    const double nm = DTSMOOTH * fi + DTSMOOTH_DIV2 * (fm + y);
    xo = y < 0. ? 0. : y;
    xn = nm < 0. ? 0. : nm;
  }
}

// The sum of v over the wavefront, in every lane: DPP row shifts and row
// broadcasts (no LDS traffic) leave it in lane 63.
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v, int rows) {
  union { double d; int w[2]; } a, b;
  a.d = v;
  b.w[0] = rows == 0xf ? __builtin_amdgcn_update_dpp(0, a.w[0], CTRL, 0xf, 0xf, true)
                       : __builtin_amdgcn_update_dpp(0, a.w[0], CTRL, 0xa, 0xf, false);
  b.w[1] = rows == 0xf ? __builtin_amdgcn_update_dpp(0, a.w[1], CTRL, 0xf, 0xf, true)
                       : __builtin_amdgcn_update_dpp(0, a.w[1], CTRL, 0xa, 0xf, false);
  return v + b.d;
}
__device__ __forceinline__ double wave_total(double v) {
  v = dpp_add<0x111>(v, 0xf);  // row_shr:1, 2, 4, 8: the row's sum in its lane 15
  v = dpp_add<0x112>(v, 0xf);
  v = dpp_add<0x114>(v, 0xf);
  v = dpp_add<0x118>(v, 0xf);
  v = dpp_add<0x142>(v, 0xa);  // row_bcast:15 into rows 1 and 3
  union { double d; int w[2]; } a, lo, hi;
  a.d = v;
  lo.w[0] = __builtin_amdgcn_readlane(a.w[0], 31);
  lo.w[1] = __builtin_amdgcn_readlane(a.w[1], 31);
  hi.w[0] = __builtin_amdgcn_readlane(a.w[0], 63);
  hi.w[1] = __builtin_amdgcn_readlane(a.w[1], 63);
  return lo.d + hi.d;
}
// Orders this wavefront's LDS writes before its LDS reads (the regions are
// private to a wavefront).
__device__ __forceinline__ void lds_wait() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Doubles of LDS of one wavefront for rows of nlon longitudes in at most maxc
// chunks: the residual of a row, whose space the chunk averages and edges take
// once the chunk sums have been read (2 maxc <= nlon unless a chunk is a single
// longitude); with lanes sharing a chunk (at most 32 chunks) 64 parts, then 32
// averages and 32 edges.
inline int wave_doubles(int nlon, int maxc) {
  const int w = nlon > 128 ? nlon : 128;
  return 2 * maxc > w ? 2 * maxc : w;
}

// NPL: longitudes per lane (nlon <= 64 NPL); lane l holds i = l + 64 t.
// LDS: the table cs[(m-1) nlon + i], sn[...] for m = 1..order, then per
// wavefront wl doubles (wave_doubles) of its own.  The launch covers nkp
// levels of each of the P.nf fields, field-major; wavefront w of block
// (r, y) takes level y W + w of that order.
// GTAB: the table is given in device memory (gtab: cos of harmonics
// 1..tord at (m-1) nlon + i, then their sin; ring_table_kernel) instead of
// being built in LDS; the LDS then holds the wavefronts' own regions only.
// The kernels below wrap this body.
// Bound by FP64 instructions and the wait for one level's loads: one level per
// wavefront with no loop over levels keeps it under 96 VGPRs (a loop with the
// next level's loads in flight let the compiler hold each longitude's chunk
// geometry across levels, 247 VGPRs, two wavefronts per SIMD).  One component
// at 0.625 deg, order 3: 83.9 us, 1.0 TB/s of its rows, before (LDS shuffles
// for the sums, a block barrier per level, four divisions by 12 per point); 44.0
// us by the profiler, 1.9 TB/s, now (40 per launch in a row of launches).  2.5 deg 21.9 -> 10.7 us, 5 deg 20.4 -> 10.6 us.
template <int NPL, bool GTAB, int MO>
__device__ __forceinline__ void ringfilter_body(const Fields &P, long plane, const Rows &R, int nlon, int nkp,
                                                int order, int oplus, double dlamda, int wl,
                                                const double *__restrict__ gtab, int tord) {
  extern __shared__ double sh[];
  const int W = blockDim.x >> 6, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r = blockIdx.x;
  const int nchnk = R.n[r];
  const int ntab = GTAB ? 0 : order * nlon;
  const double *cs = GTAB ? gtab : sh, *sn = GTAB ? gtab + (size_t)tord * nlon : sh + ntab;
  double *fx = sh + 2 * ntab + (size_t)wave * wl;
  auto trig = [&](int m, int i, double &c, double &s) {
    c = cs[(m - 1) * nlon + i];
    s = sn[(m - 1) * nlon + i];
  };
  const int kq = (int)blockIdx.y * W + wave;
  const bool live = kq < P.nf * nkp;
  const int q = live ? kq / nkp : 0, k = live ? kq - q * nkp : 0;
  const bool act = live && k < P.nlev;  // a level to filter (else the top, or none)
  const size_t off = (size_t)k * plane + R.off[r];
  double *row = P.f[q] + off;
  // :40 the interior longitudes, in flight while the table is built
  double w[NPL], v[NPL];
#pragma unroll
  for (int t = 0; t < NPL; ++t) {
    const int i = lane + 64 * t;
    w[t] = act && i < nlon ? row[2 + i] : 0.;
  }
  if (!GTAB) {
    for (int t = threadIdx.x; t < ntab; t += blockDim.x) {
      const int m = t / nlon + 1, i = t - (m - 1) * nlon;
      const double ang = (i + 1) * dlamda;
      double s, c;
      sincos(m * ang, &s, &c);
      sh[t] = c;
      sh[ntab + t] = s;
    }
    __syncthreads();
  }
  if (!live) return;
  const bool post = P.kind != POST_NONE;
  double *xr = post ? P.xnm[q] + off : row;
  if (!act) {  // the top level: spval (dt.F:407-408, duv.F:385-386, :512-513), zero (oplus.F:922-923)
    if (post) {
      const double top = P.kind == POST_OPLUS ? 0. : SPVAL;
      for (int i = lane; i < nlon + 4; i += 64) {
        row[i] = top;
        xr[i] = top;
      }
    }
    return;
  }
  // :42 their mean and :43-53 the Fourier sums of the kept harmonics (ang =
  // i dlamda, i = 1..nlon), then every sum over the wavefront
  double sum[2 * MO + 1];
  sum[0] = 0.;
#pragma unroll
  for (int t = 0; t < NPL; ++t) sum[0] += w[t];
#pragma unroll
  for (int m = 1; m <= MO; ++m) {
    sum[2 * m - 1] = sum[2 * m] = 0.;
    if (m > order) continue;
    double sa = 0., sb = 0.;
#pragma unroll
    for (int t = 0; t < NPL; ++t) {
      const int i = lane + 64 * t;
      if (i < nlon) {
        double cn, sg;
        trig(m, i, cn, sg);
        sa += w[t] * cn;
        sb += w[t] * sg;
      }
    }
    sum[2 * m - 1] = sa;
    sum[2 * m] = sb;
  }
#pragma unroll
  for (int z = 0; z <= 2 * MO; ++z)
    if (z <= 2 * order) sum[z] = wave_total(sum[z]);
  // the table is read again below: its 2 order NPL values per lane would
  // otherwise stay in registers and halve the wavefronts of a SIMD
  lds_wait();
  // :42, :53-61 the mean and the harmonic part, harmonics in ascending
  // order as the reference adds them
  const double a0 = sum[0] / nlon;
#pragma unroll
  for (int t = 0; t < NPL; ++t) v[t] = a0;
#pragma unroll
  for (int m = 1; m <= MO; ++m) {
    if (m > order) continue;
    const double am = 2. * sum[2 * m - 1] / nlon, bm = 2. * sum[2 * m] / nlon;
#pragma unroll
    for (int t = 0; t < NPL; ++t) {
      const int i = lane + 64 * t;
      if (i < nlon) {
        double cn, sg;
        trig(m, i, cn, sg);
        v[t] = v[t] + am * cn + bm * sg;
      }
    }
  }
  // :63 the residual
#pragma unroll
  for (int t = 0; t < NPL; ++t) {
    const int i = lane + 64 * t;
    if (i >= nlon) continue;
    w[t] = w[t] - v[t];
    fx[i] = w[t];
  }
  lds_wait();
  // :65-69 the chunk averages.  gsz lanes sum a chunk's parts of `per`
  // longitudes and one adds the parts up, where a few chunks of many
  // longitudes would leave most lanes idle and one lane a chain of n additions.
  const int n = nlon / nchnk;
  int gsz = nchnk <= 32 ? 64 / nchnk : 1;
  while (gsz > 1 && (gsz - 1) * (gsz - 1) >= n) --gsz;
  double *avg, *edge;
  if (gsz > 1) {
    const int per = (n + gsz - 1) / gsz;
    const int c = lane / gsz, g = lane - c * gsz;
    double s = 0.;
    if (c < nchnk) {
      const double *x = fx + c * n;
      const int m1 = min((g + 1) * per, n);
      for (int m = g * per; m < m1; ++m) s = s + x[m];
    }
    lds_wait();
    fx[lane] = s;
    lds_wait();
    avg = fx + 64;
    edge = avg + 32;
    if (lane < nchnk) {
      s = 0.;
      for (int m = 0; m < gsz; ++m) s = s + fx[lane * gsz + m];
      avg[lane] = s / n;
    }
  } else {
    avg = fx;  // chunk c's average overwrites fx[c], which is read by then (c <= c n)
    edge = fx + nchnk;
    for (int c0 = 0; c0 < nchnk; c0 += 64) {
      const int c = c0 + lane;
      double s = 0.;
      if (c < nchnk) {
        const double *x = fx + c * n;
        for (int m = 0; m < n; ++m) s = s + x[m];
      }
      lds_wait();  // all 64 chunks are read before their averages are written
      if (c < nchnk) avg[c] = s / n;
    }
  }
  lds_wait();
  // :71-83 the value at each chunk's left edge from the four neighbouring
  // averages, periodic in the chunks; a chunk's right edge is the next one's
  // left edge, term by term
  for (int c = lane; c < nchnk; c += 64) {
    int im2 = c - 2, im1 = c - 1, ip1 = c + 1;
    if (im2 < 0) im2 += nchnk;
    if (im2 < 0) im2 += nchnk;
    if (im1 < 0) im1 += nchnk;
    if (ip1 >= nchnk) ip1 -= nchnk;
    edge[c] = (-avg[im2] + 7. * avg[im1] + 7. * avg[c] - avg[ip1]) / 12.;
  }
  lds_wait();
  const double *fin = post ? P.fin[q] + off : row, *fnmi = post ? P.fnmi[q] + off : row;  // the step inputs
  // :84-101 reconstruction, the harmonic part added back, the periodic points.
  // Longitude i = lane + 64 t is point m (1-based) of chunk c; both advance by
  // 64 = q64 n + r64 per t.
  const int q64 = 64 / n, r64 = 64 - q64 * n;
  int c = lane / n, m = lane - c * n + 1;
#pragma unroll
  for (int t = 0; t < NPL; ++t) {
    const int i = lane + 64 * t;
    if (t > 0) {
      c += q64;
      m += r64;
      if (m > n) {
        m -= n;
        ++c;
      }
    }
    if (i >= nlon) continue;
    double x = w[t];
    if (c < nchnk) {  // points past nchnk * n keep their residual (:84-93 stop at nchnk * n)
      const double left = edge[c], right = edge[c + 1 < nchnk ? c + 1 : 0];
      if (oplus) {
        const double A0 = avg[c];
        const double fa = (left + right - 2. * A0) / (double)(n * n);
        const double fb = (3. * A0 - 2. * left - right) / n;
        x = fa * (3. * (m * m) - 3. * m + 1.) + fb * (2. * m - 1.) + left;
      } else {
        x = (left * (n - m) + right * m) / n;
      }
    }
    const double y = x + v[t];
    double xo = y, xn = 0.;
    if (post) {
      post_point(P.kind, y, fin[2 + i], fnmi[2 + i], xo, xn);
      xr[2 + i] = xn;
    }
    row[2 + i] = xo;
    if (t == 0 && i < 2) {
      row[nlon + 2 + i] = xo;
      if (post) xr[nlon + 2 + i] = xn;
    }
    if (64 * t + 66 > nlon && i >= nlon - 2) {
      row[i - (nlon - 2)] = xo;
      if (post) xr[i - (nlon - 2)] = xn;
    }
  }
}

template <int NPL, int MO>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(NPL <= 9 ? 4 : 2)))
ringfilter_kernel(Fields P, long plane, Rows R, int nlon, int nkp, int order, int oplus, double dlamda, int wl) {
  ringfilter_body<NPL, false, MO>(P, plane, R, nlon, nkp, order, oplus, dlamda, wl, nullptr, 0);
}

// With the table in device memory: one wavefront per block, at most 128
// VGPRs, so that four wavefronts of it fit on a SIMD beside the column
// kernels of the routines running at the same time.
template <int NPL>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(NPL <= 9 ? 4 : NPL <= 18 ? 3 : 2)))
ringfilter_gtab_kernel(Fields P, long plane, Rows R, int nlon, int nkp, int order, int oplus, double dlamda, int wl,
                       const double *__restrict__ gtab, int tord) {
  ringfilter_body<NPL, true, TGX_GLB_RING_ORDER>(P, plane, R, nlon, nkp, order, oplus, dlamda, wl, gtab, tord);
}

// The table of ringfilter_gtab_kernel: cos(m ang) and sin(m ang) of
// longitude i (ang = (i + 1) dlamda, i < nlon) for m = 1..tord, the values
// the LDS form computes.
__global__ void __launch_bounds__(64) ring_table_kernel(double *__restrict__ tab, int nlon, int tord,
                                                         double dlamda) {
  tgx_ring_table_entry(tab, nlon, tord, dlamda, blockIdx.x * blockDim.x + threadIdx.x);
}

// The same filter where the table does not fit in LDS (long rows, many
// harmonics): one wavefront per (row, level), sincos evaluated where needed.
// LDS: wm[nlon] (then the rebuilt row), fx[nlon], avg[nlon].
__global__ void __launch_bounds__(64) ringfilter_direct_kernel(double *__restrict__ f, long plane, Rows R, int nlon,
                                                        int order, int oplus, double dlamda) {
  extern __shared__ double sh[];
  double *wm = sh, *fx = sh + nlon, *avg = sh + 2 * nlon;
  const int r = blockIdx.x, k = blockIdx.y, lane = threadIdx.x;
  const int nchnk = R.n[r];
  double *row = f + (size_t)k * plane + R.off[r];
  // :40-42 the interior longitudes and their mean
  double s0 = 0.;
  for (int i = lane; i < nlon; i += 64) {
    const double w = row[2 + i];
    fx[i] = w;
    s0 += w;
  }
  const double a0 = wave_sum(s0) / nlon;
  // :43-53 Fourier coefficients of the kept harmonics (ang = i dlamda, i = 1..nlon)
  double a[kMaxOrder + 1], b[kMaxOrder + 1];
  for (int m = 1; m <= order; ++m) {
    double sa = 0., sb = 0.;
    for (int i = lane; i < nlon; i += 64) {
      const double ang = (i + 1) * dlamda;
      double sn, cn;
      sincos(m * ang, &sn, &cn);
      sa += fx[i] * cn;
      sb += fx[i] * sn;
    }
    a[m] = 2. * wave_sum(sa) / nlon;
    b[m] = 2. * wave_sum(sb) / nlon;
  }
  // :55-63 the harmonic part and the residual
  for (int i = lane; i < nlon; i += 64) {
    const double ang = (i + 1) * dlamda;
    double v = a0;
    for (int m = 1; m <= order; ++m) {
      double sn, cn;
      sincos(m * ang, &sn, &cn);
      v = v + a[m] * cn + b[m] * sn;
    }
    wm[i] = v;
    fx[i] = fx[i] - v;
  }
  __syncthreads();
  // :65-69 chunk averages, each summed in longitude order
  const int n = nlon / nchnk;
  for (int c = lane; c < nchnk; c += 64) {
    double s = 0.;
    for (int m = 0; m < n; ++m) s = s + fx[c * n + m];
    avg[c] = s / n;
  }
  __syncthreads();
  // :71-97 reconstruction from the four neighbouring chunk averages; the
  // rebuilt value of longitude i replaces wm[i], which only this lane reads
  for (int i = lane; i < nlon; i += 64) {
    const int c = i / n;
    double x = fx[i];
    if (c < nchnk) {  // points past nchnk * n keep their residual (:84-93 stop at nchnk * n)
      const int m = i - c * n + 1;
      const int im2 = (c - 2 + 2 * nchnk) % nchnk, im1 = (c - 1 + nchnk) % nchnk;
      const int ip1 = (c + 1) % nchnk, ip2 = (c + 2) % nchnk;
      const double A0 = avg[c];
      const double left = (-avg[im2] + 7. * avg[im1] + 7. * A0 - avg[ip1]) / 12.;
      const double right = (-avg[im1] + 7. * A0 + 7. * avg[ip1] - avg[ip2]) / 12.;
      if (oplus) {
        const double fa = (left + right - 2. * A0) / (double)(n * n);
        const double fb = (3. * A0 - 2. * left - right) / n;
        x = fa * (3. * (m * m) - 3. * m + 1.) + fb * (2. * m - 1.) + left;
      } else {
        x = (left * (n - m) + right * m) / n;
      }
    }
    wm[i] = x + wm[i];
    row[2 + i] = wm[i];
  }
  __syncthreads();
  // :99-101 periodic points
  if (lane == 0) row[0] = wm[nlon - 2];
  if (lane == 1) row[1] = wm[nlon - 1];
  if (lane == 2) row[nlon + 2] = wm[0];
  if (lane == 3) row[nlon + 3] = wm[1];
}

// Whether the table and the rows of 2 to kWaves wavefronts fit in a block's LDS;
// if not, the launcher filters with ringfilter_direct_kernel (one field, no post
// pass).  A table for one wavefront's level takes as many sincos as that filter
// and leaves one wavefront per block: 1152 longitudes, order 3, 113 levels 325 us
// direct and 429, 1536, order 2, 397 and 468.  With two wavefronts the table wins
// (1024, order 3, 113 levels 176 us; 355 for a table per three levels of one).
inline bool table_fits(int nlon, int order, int wl, int *waves) {
  const size_t tab = sizeof(double) * 2 * (size_t)order * nlon, per = sizeof(double) * wl;
  int W = kWaves;
  while (W > 2 && tab + W * per > kLdsMax) W >>= 1;
  if (waves) *waves = W;
  return tab + W * per <= kLdsMax;
}

template <int NPL>
int launch(const Fields &P, int nkp, long plane, int nrows, const Rows &R, int nlon, int order, int oplus,
           double dlamda, const double *gtab, int tord, hipStream_t s) {
  int W = 1, maxc = 1;
  for (int r = 0; r < nrows; ++r) maxc = R.n[r] > maxc ? R.n[r] : maxc;
  const int wl = wave_doubles(nlon, maxc);
  if (gtab) {
    // one wavefront per block and level: small blocks (4.6 KB of LDS at 576
    // longitudes) that find room beside the column kernels of the other
    // routines running at the same time
    const size_t lds = sizeof(double) * wl;
    const unsigned ny = (unsigned)((long)P.nf * nkp);
    hipLaunchKernelGGL((ringfilter_gtab_kernel<NPL>), dim3((unsigned)nrows, ny), dim3(64), lds, s, P, plane, R, nlon,
                       nkp, order, oplus, dlamda, wl, gtab, tord);
  } else if (!table_fits(nlon, order, wl, &W)) {
    if (P.nf != 1 || P.kind != POST_NONE || nkp != P.nlev)
      return tgx_set_error(TGX_ERR_ARG, "ring filter: fused post pass needs the LDS table (nlon %d, order %d)",
                           nlon, order);
    hipLaunchKernelGGL(ringfilter_direct_kernel, dim3((unsigned)nrows, (unsigned)nkp), dim3(64),
                       sizeof(double) * 3 * (size_t)nlon, s, P.f[0], plane, R, nlon, order, oplus, dlamda);
  } else {
    const size_t lds = sizeof(double) * (2 * (size_t)order * nlon + (size_t)W * wl);
    const unsigned ny = (unsigned)(((long)P.nf * nkp + W - 1) / W);
    if (order <= 3)  // the model's orders: seven sums held instead of seventeen
      hipLaunchKernelGGL((ringfilter_kernel<NPL, 3>), dim3((unsigned)nrows, ny), dim3(64 * W), lds, s, P, plane, R, nlon,
                         nkp, order, oplus, dlamda, wl);
    else
      hipLaunchKernelGGL((ringfilter_kernel<NPL, kMaxOrder>), dim3((unsigned)nrows, ny), dim3(64 * W), lds, s, P,
                         plane, R, nlon, nkp, order, oplus, dlamda, wl);
  }
  TGX_HIP(hipGetLastError());
  return 0;
}

inline int launch_any(const Fields &P, int nkp, long plane, int nrows, const Rows &R, int nlon, int order,
                      int oplus, double dlamda, const double *gtab, int tord, hipStream_t s) {
  if (nlon <= 64 * 2) return launch<2>(P, nkp, plane, nrows, R, nlon, order, oplus, dlamda, gtab, tord, s);
  if (nlon <= 64 * 3) return launch<3>(P, nkp, plane, nrows, R, nlon, order, oplus, dlamda, gtab, tord, s);
  if (nlon <= 64 * 5) return launch<5>(P, nkp, plane, nrows, R, nlon, order, oplus, dlamda, gtab, tord, s);
  if (nlon <= 64 * 9) return launch<9>(P, nkp, plane, nrows, R, nlon, order, oplus, dlamda, gtab, tord, s);
  if (nlon <= 64 * 18) return launch<18>(P, nkp, plane, nrows, R, nlon, order, oplus, dlamda, gtab, tord, s);
  return launch<32>(P, nkp, plane, nrows, R, nlon, order, oplus, dlamda, gtab, tord, s);
}

}  // namespace ring
}  // namespace tgx

namespace {
// Validates a launch of nrows rows (host arrays rowoff, nchnk, at most
// TGX_RING_MAX_ROWS) and launches it.
int launch_rows(const tgx::ring::Fields &P, int nkp, long plane, int nrows, const long *rowoff, const int *nchnk,
                int nlon, int order, int oplus, double dlamda, hipStream_t s, const double *gtab = nullptr,
                int tord = 0) {
  if (nrows <= 0 || nkp <= 0 || P.nf <= 0) return 0;
  if (nrows > TGX_RING_MAX_ROWS) return tgx_set_error(TGX_ERR_ARG, "ring filter: %d rows > %d", nrows, TGX_RING_MAX_ROWS);
  if (nlon < 4 || nlon > TGX_RING_MAX_NLON || order < 0 || order > tgx::ring::kMaxOrder || order >= nlon)
    return tgx_set_error(TGX_ERR_ARG, "ring filter: nlon %d (4..%d) or order %d (0..%d, < nlon)", nlon,
                         TGX_RING_MAX_NLON, order, tgx::ring::kMaxOrder);
  tgx::ring::Rows R;
  for (int r = 0; r < nrows; ++r) {
    if (nchnk[r] < 1 || nchnk[r] > nlon)
      return tgx_set_error(TGX_ERR_ARG, "ring filter: %d chunks for %d longitudes", nchnk[r], nlon);
    R.off[r] = rowoff[r];
    R.n[r] = nchnk[r];
  }
  if (gtab && (order > tord || order > TGX_GLB_RING_ORDER))
    return tgx_set_error(TGX_ERR_ARG, "ring filter: order %d beyond the table's %d", order, tord);
  return tgx::ring::launch_any(P, nkp, plane, nrows, R, nlon, order, oplus, dlamda, gtab, tord, s);
}

// The latitudes next to each pole that the chunk table filters
// (ringfilter.F:23-34), as row offsets in the level-plane layout of
// tgx_step.h (latitude lat is row lat + 1 of the nlat + 4 rows).
int polar_rows(int nlat, int ld, int nlat_filter, const int *chunk, long *off, int *nc) {
  int nrows = 0;
  for (int lat = 1; lat <= nlat; ++lat) {
    int c = 0;
    if (lat <= nlat_filter) c = chunk[lat - 1];
    else if (lat >= nlat - nlat_filter + 1) c = chunk[nlat - lat];
    if (c == 0) continue;
    off[nrows] = (long)(lat + 1) * ld;
    nc[nrows] = c;
    ++nrows;
  }
  return nrows;
}

tgx::ring::Fields one_field(double *f, int nk) {
  tgx::ring::Fields P = {};
  P.f[0] = f;
  P.nf = 1;
  P.nlev = nk;
  P.kind = tgx::ring::POST_NONE;
  return P;
}
}  // namespace

// Launcher of the host drop-in: nrows rows of nk levels of one field.
extern "C" int tgx_launch_ringfilter(double *f, int nk, long plane, int nrows, const long *rowoff,
                                     const int *nchnk, int nlon, int order, int oplus, double dlamda,
                                     hipStream_t s) {
  return launch_rows(one_field(f, nk), nk, plane, nrows, rowoff, nchnk, nlon, order, oplus, dlamda, s);
}

extern "C" int tgx_ringfilter_dev(double *f, int nk, int nlon, int nlat, int ld, int order, int oplus,
                                  double dlamda, int nlat_filter, const int *chunk, void *stream) {
  if (!f || nk <= 0 || nlat <= 0 || ld < nlon + 4 || nlat_filter < 0 || nlat_filter > TGX_RING_MAX_ROWS / 2 ||
      (nlat_filter > 0 && !chunk))
    return tgx_set_error(TGX_ERR_ARG, "tgx_ringfilter_dev: bad arguments (nk %d nlon %d nlat %d ld %d nlat_filter %d)",
                         nk, nlon, nlat, ld, nlat_filter);
  long off[TGX_RING_MAX_ROWS];
  int nc[TGX_RING_MAX_ROWS];
  const int nrows = polar_rows(nlat, ld, nlat_filter, chunk, off, nc);
  return launch_rows(one_field(f, nk), nk, (long)ld * (nlat + 4), nrows, off, nc, nlon, order, oplus, dlamda,
                     (hipStream_t)stream);
}

// The cos/sin table of tgx_ringfilter_post_dev (harmonics 1..tord of nlon
// longitudes, 2 tord nlon doubles at tab), on the stream.
extern "C" int tgx_ring_table_dev(double *tab, int nlon, int tord, double dlamda, hipStream_t s) {
  if (!tab || nlon < 4 || nlon > TGX_RING_MAX_NLON || tord < 1 || tord > tgx::ring::kMaxOrder)
    return tgx_set_error(TGX_ERR_ARG, "ring filter table: nlon %d (4..%d), order %d (1..%d)", nlon, TGX_RING_MAX_NLON,
                         tord, tgx::ring::kMaxOrder);
  const int n = tord * nlon;
  hipLaunchKernelGGL(tgx::ring::ring_table_kernel, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, s, tab, nlon,
                     tord, dlamda);
  TGX_HIP(hipGetLastError());
  return 0;
}

// The ring filters of one global routine in one launch: the nf (<= 4) fields
// f[q] on their polar latitudes, levels 0..nlev-1, each filtered value then
// passed through the routine's post pass `kind` (tgx::ring::PostKind) with
// the step inputs fin[q], fnmi[q] into f[q] and xnm[q]; with a post pass and
// nlev < nk, the top level nlev is set as the routine sets it.  The periodic
// points of the filtered rows are rewritten; the other latitudes are not
// touched.  gtab: the table of tgx_ring_table_dev for harmonics 1..tord
// (order <= tord), filled on the same stream.  Used by the global routines
// (step_api.cpp).
extern "C" int tgx_ringfilter_post_dev(int nf, double *const *f, double *const *xnm, const double *const *fin,
                                       const double *const *fnmi, int kind, int nlev, int nk, int nlon, int nlat,
                                       int ld, int order, int oplus, double dlamda, int nlat_filter,
                                       const int *chunk, const double *gtab, int tord, hipStream_t s) {
  if (nf < 1 || nf > 4 || kind < tgx::ring::POST_NONE || kind > tgx::ring::POST_OPLUS || nlev < 1 || nlev > nk ||
      (kind != tgx::ring::POST_NONE && nk - nlev > 1) || nlat <= 0 || ld < nlon + 4 || nlat_filter < 0 ||
      nlat_filter > TGX_RING_MAX_ROWS / 2 || (nlat_filter > 0 && !chunk) || !gtab)
    return tgx_set_error(TGX_ERR_ARG, "ring filter + post: bad arguments (nf %d kind %d nlev %d nk %d)", nf, kind,
                         nlev, nk);
  tgx::ring::Fields P = {};
  for (int q = 0; q < nf; ++q) {
    P.f[q] = f[q];
    if (kind != tgx::ring::POST_NONE) {
      P.xnm[q] = xnm[q];
      P.fin[q] = fin[q];
      P.fnmi[q] = fnmi[q];
    }
  }
  P.nf = nf;
  P.nlev = nlev;
  P.kind = kind;
  long off[TGX_RING_MAX_ROWS];
  int nc[TGX_RING_MAX_ROWS];
  const int nrows = polar_rows(nlat, ld, nlat_filter, chunk, off, nc);
  return launch_rows(P, kind != tgx::ring::POST_NONE ? nk : nlev, (long)ld * (nlat + 4), nrows, off, nc, nlon,
                     order, oplus, dlamda, s, gtab, tord);
}
