// The global grid's passes around the column kernels of the larger grids: the
// periodic points of the outputs (mp_periodic_f3d), the rows across the poles
// of O+ between sub-cycles, and the halos of an input field (mk_polelat.F,
// mp_periodic_f4d).  The post passes are the column kernels', the ring filter
// launch's and comp_post_block's; the block kernels of the smaller grids write
// the periodic points themselves.  Level planes as in tgx_step.h; the
// elementwise passes take one thread per (point, level), the longitudes
// fastest.
#include <hip/hip_runtime.h>

#include "../../include/tgx.h"
#include "../../include/tgx_global.h"
#include "tgx_common.h"

namespace tgx {
namespace glb {

struct Dims {
  int nk, nlon, nlat, ld;
  size_t plane;  // ld * (nlat + 4)
};

// mp_periodic_f3d on the interior latitudes of up to eight fields: thread
// per (periodic point, interior latitude, level, field).
struct Periodic {
  double *f[8];
  int n, nk;
};

__global__ void __launch_bounds__(256) periodic_kernel(Dims D, Periodic P) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long per = 4L * D.nlat * P.nk;
  if (t >= per * P.n) return;
  const int q = (int)(t / per);
  long r = t - (long)q * per;
  const int k = (int)(r / (4L * D.nlat));
  r -= (long)k * 4L * D.nlat;
  const int j = 2 + (int)(r / 4), c = (int)(r & 3);
  const int dst = c == 0 ? 0 : c == 1 ? 1 : c == 2 ? D.nlon + 2 : D.nlon + 3;
  const int src = c == 0 ? D.nlon : c == 1 ? D.nlon + 1 : c == 2 ? 2 : 3;
  double *row = P.f[q] + (size_t)k * D.plane + (size_t)j * D.ld;
  row[dst] = row[src];
}

// The rows across the poles of `dst` from those of `src` (O+ between
// sub-cycles): thread per (column, ghost row, level).
__global__ void __launch_bounds__(256) ghost_rows_kernel(Dims D, const double *__restrict__ src,
                                                         double *__restrict__ dst) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int nlond = D.nlon + 4;
  if (t >= 4L * nlond * D.nk) return;
  const int k = (int)(t / (4L * nlond));
  const long r = t - (long)k * 4L * nlond;
  const int g = (int)(r / nlond), i = (int)(r - (long)g * nlond);
  const int j = g < 2 ? g : D.nlat + g;  // 0, 1, nlat+2, nlat+3
  const size_t p = (size_t)k * D.plane + (size_t)j * D.ld + i;
  dst[p] = src[p];
}

// tgx_glb_halos: periodic points of the interior rows and the rows across
// the poles, thread per (column, row to fill, level); the pole rows read the
// interior columns of interior rows only, so the two kinds of writes are
// independent.
__global__ void __launch_bounds__(256) halos_kernel(Dims D, double *__restrict__ f, double sign) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int nlond = D.nlon + 4;
  const long nper = 4L * D.nlat, npole = 4L * nlond;
  if (t >= (nper + npole) * D.nk) return;
  const int k = (int)(t / (nper + npole));
  long r = t - (long)k * (nper + npole);
  double *pl = f + (size_t)k * D.plane;
  if (r < nper) {
    const int j = 2 + (int)(r / 4), c = (int)(r & 3);
    const int dst = c == 0 ? 0 : c == 1 ? 1 : c == 2 ? D.nlon + 2 : D.nlon + 3;
    const int src = c == 0 ? D.nlon : c == 1 ? D.nlon + 1 : c == 2 ? 2 : 3;
    pl[(size_t)j * D.ld + dst] = pl[(size_t)j * D.ld + src];
    return;
  }
  r -= nper;
  const int g = (int)(r / nlond), i = (int)(r - (long)g * nlond);
  // latitude 0 <- 1, -1 <- 2, nlat+1 <- nlat, nlat+2 <- nlat-1 (rows j = lat + 1)
  const int jnew = g == 0 ? 1 : g == 1 ? 0 : g == 2 ? D.nlat + 2 : D.nlat + 3;
  const int jold = g == 0 ? 2 : g == 1 ? 3 : g == 2 ? D.nlat + 1 : D.nlat;
  const int isrc = ((i - 2 + D.nlon / 2) % D.nlon + D.nlon) % D.nlon + 2;
  pl[(size_t)jnew * D.ld + i] = sign * pl[(size_t)jold * D.ld + isrc];
}

inline unsigned nblocks(long n) { return (unsigned)((n + 255) / 256); }

Dims dims_of(const tgx_ng_grid *g) {
  Dims D;
  D.nk = g->nk;
  D.nlon = g->nlon;
  D.nlat = g->nlat;
  D.ld = g->ld;
  D.plane = (size_t)g->ld * (size_t)(g->nlat + 4);
  return D;
}

int periodic(const Dims &D, double *const *f, int n, int nk, hipStream_t s) {
  Periodic P = {};
  for (int q = 0; q < n; ++q) P.f[q] = f[q];
  P.n = n;
  P.nk = nk;
  hipLaunchKernelGGL(periodic_kernel, dim3(nblocks(4L * D.nlat * nk * n)), dim3(256), 0, s, D, P);
  TGX_HIP(hipGetLastError());
  return 0;
}

}  // namespace glb
}  // namespace tgx

using namespace tgx::glb;

// What remains of a global routine's larger-grid form after its post pass
// (the column kernel's, the ring filter launch's and, for comp,
// comp_post_block's): which 0 dt, 1 duv, 2 minor species N2D and Ar, 3 minor
// species NO and N4S, 4 O+ sub-step (op_o, nm_o: its outputs, whose rows
// across the poles take those of in->op / in->op_nm), 5 comp.  The periodic
// points of the outputs on every interior latitude.
extern "C" int tgx_glb_post(int which, const tgx_ng_grid *g, const tgx_ng_fields *in, const tgx_ng_out *out,
                            double *op_o, double *nm_o, hipStream_t s) {
  if (which < 0 || which > 5) return tgx_set_error(TGX_ERR_ARG, "tgx_glb_post: unknown pass %d", which);
  const Dims D = dims_of(g);
  // mp_periodic_f3d of every output the pass wrote
  double *per[8];
  int n = 0;
  switch (which) {
    case 0: per[n++] = out->tn; per[n++] = out->tn_nm; break;
    case 1: per[n++] = out->un; per[n++] = out->vn; per[n++] = out->un_nm; per[n++] = out->vn_nm; break;
    case 2: per[n++] = out->n2d; per[n++] = out->n2d_nm; per[n++] = out->ar; per[n++] = out->ar_nm; break;
    case 3: per[n++] = out->no; per[n++] = out->no_nm; per[n++] = out->n4s; per[n++] = out->n4s_nm; break;
    case 4: per[n++] = op_o; per[n++] = nm_o; break;
    default:
      per[n++] = out->o2; per[n++] = out->o1; per[n++] = out->he;
      per[n++] = out->o2_nm; per[n++] = out->o1_nm; per[n++] = out->he_nm;
  }
  if (int rc = periodic(D, per, n, D.nk, s)) return rc;
  if (which == 1) {  // the lower-boundary winds (duv.F:473-500)
    double *per2[4] = {out->ulbc, out->vlbc, out->ulbc_nm, out->vlbc_nm};
    if (int rc = periodic(D, per2, 4, 1, s)) return rc;
  }
  if (which == 4) {
    hipLaunchKernelGGL(ghost_rows_kernel, dim3(nblocks(4L * (D.nlon + 4) * D.nk)), dim3(256), 0, s, D, in->op, op_o);
    hipLaunchKernelGGL(ghost_rows_kernel, dim3(nblocks(4L * (D.nlon + 4) * D.nk)), dim3(256), 0, s, D, in->op_nm,
                       nm_o);
    TGX_HIP(hipGetLastError());
  }
  return 0;
}

extern "C" int tgx_glb_halos(double *f, int nk, int nlon, int nlat, int ld, double sign, void *stream) {
  if (!f || nk < 1 || nlon < 4 || (nlon & 1) || nlat < 4 || ld < nlon + 4)
    return tgx_set_error(TGX_ERR_ARG, "tgx_glb_halos: bad arguments (nk %d nlon %d (even) nlat %d ld %d)", nk, nlon,
                         nlat, ld);
  Dims D;
  D.nk = nk;
  D.nlon = nlon;
  D.nlat = nlat;
  D.ld = ld;
  D.plane = (size_t)ld * (size_t)(nlat + 4);
  const long n = (4L * nlat + 4L * (nlon + 4)) * nk;
  hipLaunchKernelGGL(halos_kernel, dim3(nblocks(n)), dim3(256), 0, (hipStream_t)stream, D, f, sign);
  TGX_HIP(hipGetLastError());
  return 0;
}
